// Shared between the gfx950 attention kernels and their launchers (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include <type_traits>

#include "../../include/mi355x_fattn.h"

#define FATTN_QK8_0 32
#define FATTN_Q8_0_BYTES 34
#define FATTN_IS_BLOCK_TYPE(t) ((t) == MI355X_TYPE_Q8_0 || (t) == MI355X_TYPE_Q4_0 || (t) == MI355X_TYPE_Q4_1 || (t) == MI355X_TYPE_Q5_0 || (t) == MI355X_TYPE_Q5_1)

// Unsigned division by a number fixed on the host, as multiply and shift (Granlund and Montgomery, "Division by invariant
// integers using multiplication", 1994): n / d = (mulhi(n, m) + n) >> s for n < 2^31.
struct FastDiv {
    uint32_t d, m, s;
};
static inline FastDiv fast_div(uint32_t d) {
    FastDiv f;
    f.d = d;
    f.s = 0;
    if (d > 1) f.s = 32 - (uint32_t)__builtin_clz(d - 1);       // the smallest s with 2^s >= d
    f.m = d ? (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << f.s) - d)) / d + 1) : 0;
    return f;
}
static __host__ __device__ __forceinline__ uint32_t divide(uint32_t n, const FastDiv & f) { return ((uint32_t)(((uint64_t)n * f.m) >> 32) + n) >> f.s; }

// Everything a kernel needs about one FLASH_ATTN_EXT node, by value.
struct FattnArgs {
    const char * q;      // F32  [D, Nq, Hq, B]
    const char * k;      // K/V storage type [D, Nkv, Hkv, Bk]
    const char * v;
    const char * mask;   // F16 [>=Nkv, >=Nq, Hm, Bm] or nullptr
    float *      dst;    // F32 [D, Hq, Nq, B] contiguous

    int32_t D, Nq, Hq, B, Nkv, Hkv, Bk;
    int32_t Dv;          // elements of a q row and of a dst row; = D, except when the tile kernel runs a head size it has no
                         // form for on f16 copies of K/V whose rows are zero-padded to D (64 or 128): then the real head size
    int32_t gqa;         // Hq / Hkv
    int32_t bq;          // B / Bk
    int32_t q_chunks;    // decode kernel: 16-row chunks of the Nq * gqa query rows that share a KV head
    int32_t Hm, Bm;      // mask broadcast extents
    int32_t masked;      // the call has a mask (planning looks here: `mask` may still be null when a call is only being sized)

    int64_t nbq1, nbq2, nbq3;
    int64_t nbk1, nbk2, nbk3;
    int64_t nbv1, nbv2, nbv3;
    int64_t nbm1, nbm2, nbm3;

    float scale;         // already divided by logit_softcap when that is non-zero
    float softcap;
    float max_bias, m0, m1;
    int32_t n_head_log2;

    int32_t aligned16;   // q, k and v bases and strides are all multiples of 16 bytes
    int32_t q_aligned16; // q alone
    int32_t kv_aligned16; // k and v alone
    int32_t kv_aligned4;
    int32_t kv_aligned2;  // k and v: base and strides even (what the Q8_0 halfword reads need)
    int32_t mask_al8;    // mask base and strides are multiples of 8 bytes
    int32_t mask_al4;    // ... of 4 bytes
    int32_t n_cus;       // compute units of the device
    int32_t tile_variant; // 0, or 16 * key_split + query_blocks forced by the caller

    // split-KV
    int32_t n_splits;
    int32_t keys_per_split;
    float * part_acc;    // [rows, n_splits, D]  unnormalised accumulators
    float * part_ml;     // [rows, n_splits, 2]  running max, running sum
    // nullptr: the partials are merged by fattn_merge_kernel, a launch of its own.  Else one counter per set of
    // workgroups that share output rows (zero between launches): every workgroup adds one when its partials are out, and
    // the one that finds the set complete merges the rows itself and leaves the counter at zero again.
    unsigned * counters;
    // decode kernel: filled in by its launcher
    FastDiv by_splits, by_chunks, by_hkv, by_gqa, by_bq, by_hm, by_bm;
};

// kernel<<<grid, block, lds, stream>>>(args ...) in one call of the runtime: the launch expression, and hipLaunchKernelGGL with it, first
// hands the configuration over in a call of its own that the kernel's host stub takes back in another, 2.43 us of host time a launch
// against 2.23 of this (a stream that is not waited for, arguments of 80 bytes).  Errors are the runtime's last error, as behind those.
template <typename... P, typename... A>
static inline void fattn_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, const A &... args) {
    auto go = [&](P... p) {
        void * at[] = {(void *)&p...};
        (void)hipLaunchKernel((const void *)kernel, grid, block, at, lds, stream);
    };
    go(args...);
}

// Arguments S of a short launch whose first 56 bytes are in scalar registers when a wave starts (the kernel's first seven 64-bit
// parameters, by the compiler's -amdgpu-kernarg-preload-count; a structure is always read from memory): what a kernel's first
// requests are made from goes there, and the rest is on its way meanwhile.  A load of the arguments takes 565 cycles in a stream of
// launches and 200 in a graph; a chain of launches of 4.4 us each, 160 workgroups, 4.65 us with a structure and 4.39 like this.  Launches
// that do not wait for more than their arguments gain nothing by it (0.15 us longer in a graph).
template <typename S> struct ArgTail {
    uint32_t w[(sizeof(S) - 56) / 4];
};
#define FATTN_HEAD_PARAMS const uint64_t h0, const uint64_t h1, const uint64_t h2, const uint64_t h3, const uint64_t h4, const uint64_t h5, const uint64_t h6
#define FATTN_HEAD_ARGS h0, h1, h2, h3, h4, h5, h6
// (what the compiler knows of pointers among a kernel's parameters and has to be told of ones put together from numbers: device memory)
template <typename T> static __device__ __forceinline__ void fattn_global(T *& p) { p = (T *)(__attribute__((address_space(1))) T *)(uint64_t)p; }
template <typename S>
static __device__ __forceinline__ S fattn_join(FATTN_HEAD_PARAMS, const ArgTail<S> & tail) {
    struct {
        uint64_t   head[7];
        ArgTail<S> tail;
    } both = {{h0, h1, h2, h3, h4, h5, h6}, tail};
    S s;
    __builtin_memcpy(&s, &both, sizeof(S));
    s.pointers([](auto &... p) { (fattn_global(p), ...); });
    return s;
}
template <typename S>
static inline void fattn_launch_head(void (*kernel)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, ArgTail<S>), dim3 grid, dim3 block,
                                     size_t lds, hipStream_t stream, const S & s) {
    static_assert(sizeof(S) > 56 && sizeof(S) % 8 == 0 && sizeof(S) <= 112, "seven numbers and a tail");
    const char * p = (const char *)&s;
    void * at[] = {(void *)p, (void *)(p + 8), (void *)(p + 16), (void *)(p + 24), (void *)(p + 32), (void *)(p + 40), (void *)(p + 48), (void *)(p + 56)};
    (void)hipLaunchKernel((const void *)kernel, grid, block, at, lds, stream);
}

// Workgroups that use more than 64 KiB of dynamic LDS need hipFuncAttributeMaxDynamicSharedMemorySize raised, and that
// attribute belongs to the (kernel, device) pair: `done` is the launcher's own record per kernel instantiation, one bit
// per device.  Racing callers at worst set the attribute twice.
static inline hipError_t fattn_allow_lds(const void * kernel, int lds_bytes, std::atomic<uint64_t> & done) {
    if (lds_bytes <= 64 * 1024) return hipSuccess;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;      // devices past 63: set on every launch
    if (bit && (done.load(std::memory_order_relaxed) & bit)) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e == hipSuccess && bit) done.fetch_or(bit, std::memory_order_relaxed);
    return e;
}

static __device__ __forceinline__ float fattn_slope(const FattnArgs & a, int h) {
    if (a.max_bias <= 0.0f) return 1.0f;
    return h < a.n_head_log2 ? powf(a.m0, (float)(h + 1)) : powf(a.m1, (float)(2 * (h - a.n_head_log2) + 1));
}

// A load marked non-temporal, for data that a launch reads once: it leaves the rest of L2 alone and streams faster (a
// read-only sweep of 2 GiB reaches 7.0-7.1 TB/s with it against 5.7-6.2 TB/s with plain loads; a copy gains 5%).  T is
// a scalar or an ext_vector_type.  Not for lines that the same launch touches again (64-byte pieces of mask rows and
// per-lane pieces of block rows were slower with it), nor for a source that the previous launch has just written (the
// F32 -> f16 pass over fresh K/V lost 4% with it).
template <typename T>
static __device__ __forceinline__ T stream_load(const void * p) { return __builtin_nontemporal_load((const T *)p); }

// a * b + c with the product and the sum each rounded to f32, as two graph nodes (or two scalar statements) round them.
// hipcc contracts a * b + c into one fused multiply-add by default, also when it is spelled __fadd_rn(__fmul_rn(a, b), c):
// those inline as contractible operations.  Only operations compiled under "contract(off)" stay apart.
static __device__ __forceinline__ float mul_then_add(float a, float b, float c) {
#pragma clang fp contract(off)
    const float p = a * b;
    return p + c;
}

static __device__ __forceinline__ float h2f_bits(uint16_t h) {
    return (float)__builtin_bit_cast(_Float16, h);
}

// ---- DPP wavefront reductions -------------------------------------------------------
// Butterfly sums over aligned groups of lanes; every lane of a group ends with the total.
template <int CTRL>
static __device__ __forceinline__ float dpp_mov(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

static __device__ __forceinline__ float xor_shuffle(float x, int mask) {
    return __shfl_xor(x, mask, 64);
}

template <int GROUP>
static __device__ __forceinline__ float group_sum(float x) {
    static_assert(GROUP == 4 || GROUP == 8 || GROUP == 16 || GROUP == 32 || GROUP == 64, "group size");
    x += dpp_mov<0xB1>(x);                        // quad_perm [1,0,3,2]
    x += dpp_mov<0x4E>(x);                        // quad_perm [2,3,0,1]
    if (GROUP >= 8)  x += dpp_mov<0x141>(x);      // row_half_mirror: pairs the two quads of 8 lanes
    if (GROUP >= 16) x += dpp_mov<0x140>(x);      // row_mirror: pairs the two halves of a row of 16
    if (GROUP >= 32) x += xor_shuffle(x, 16);
    if (GROUP >= 64) x += xor_shuffle(x, 32);
    return x;
}

// values of the other lanes of a quad (4 lanes): lane ^ 1, lane ^ 2, lane k
static __device__ __forceinline__ uint32_t quad_swap1(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true); }
static __device__ __forceinline__ uint32_t quad_swap2(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, true); }
static __device__ __forceinline__ float quad_broadcast(float x, int k) {          // k: a constant after unrolling
    switch (k) {
        case 0:  return dpp_mov<0x00>(x);
        case 1:  return dpp_mov<0x55>(x);
        case 2:  return dpp_mov<0xAA>(x);
        default: return dpp_mov<0xFF>(x);
    }
}

// 16 bytes a lane from `base` (the same for every lane) + off to LDS address `to` + 16 * lane.  As asm because the compiler's own
// bookkeeping of such loads makes every LDS read that may alias them wait.  It places no wait states around asm either, and a
// load must not read an SGPR within five of the vector instruction that wrote it, as is the readlane of a spilled base where
// scalar registers are short.  MOVE: the base goes through a scalar move, which may read it at once.  Without it, for kernels
// that keep their bases in scalar registers: tests/test_kernel_resources.py fails if one of those loads has such a write close
// before it.  (The pipelined kernel's forms without a mask spill none - the three masked ones 21 to 24 scalar registers - and a move in
// their step, wherever it stands, costs a wave that is alone on its SIMD more than it looks: six layers of Whisper base 119.5 us, with a move ahead of each load 121, with one a step 124 to 130.)
template <bool MOVE>
static __device__ __forceinline__ void load_to_lds16(uint64_t base, uint32_t off, uint32_t to) {
    // (the readfirstlanes say that the addresses are uniform and cost nothing where the register allocator knows)
    const uint64_t p = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base);
    const uint32_t t = (uint32_t)__builtin_amdgcn_readfirstlane((int)to);
    if constexpr (MOVE) {
        uint64_t q;
        asm volatile("s_mov_b64 %0, %2\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0"
                     : "=&s"(q) : "v"(off), "s"(p), "s"(t) : "memory", "m0");
    } else {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(p), "s"(t) : "memory", "m0");
    }
}

// Workgroups of a masked call differ in length (causal rows, padded sequences): an XCD's are ordered from the last query tile to the
// first, and every second group of n_cus / 8 - the ones that join the group before on its CUs - backwards, so that a CU's two add
// up to about the same.  In the tile-wise kernel, us a layer without it, without the turn and with it: 2048 causal tokens, 32 heads of
// 128 89, 79 and 76; 16 heads of 64 56 and 51 (plain and with it).  For grids of whole heads an XCD (per = workgroups of one).
static __device__ __forceinline__ void masked_order(int per, int n_qtiles, int n_cus, int & qt, int & pair) {
    const int cus = n_cus >= 8 ? n_cus / 8 : 32, heads = per / n_qtiles;
    int i = blockIdx.x / 8;
    const int seg = i / cus * cus;
    if ((i / cus) & 1) i = seg + min(cus, per - seg) - 1 - (i - seg);
    qt   = n_qtiles - 1 - i / heads;
    pair = (int)(blockIdx.x % 8) * heads + i % heads;
}

// lane l's and lane (l ^ 32)'s values, the lower lane's first, without the LDS crossbar (whose traffic would blur the waits of
// a loop, and whose addresses cost registers)
static __device__ __forceinline__ float2 both_halves(float x) {
    uint32_t a = __float_as_uint(x), b = a;
    asm volatile("" : "+v"(b));                    // (the swap of a value with itself is folded wrongly)
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
static __device__ __forceinline__ float max_of_halves(float x) {
    const float2 v = both_halves(x);
    return fmaxf(v.x, v.y);
}
static __device__ __forceinline__ float sum_of_halves(float x) {
    const float2 v = both_halves(x);
    return v.x + v.y;
}

template <int GROUP>
static __device__ __forceinline__ float group_max(float x) {
    x = fmaxf(x, dpp_mov<0xB1>(x));
    x = fmaxf(x, dpp_mov<0x4E>(x));
    if (GROUP >= 8)  x = fmaxf(x, dpp_mov<0x141>(x));
    if (GROUP >= 16) x = fmaxf(x, dpp_mov<0x140>(x));
    if (GROUP >= 32) x = fmaxf(x, xor_shuffle(x, 16));
    if (GROUP >= 64) x = fmaxf(x, xor_shuffle(x, 32));
    return x;
}

// ---- merging split-KV partials ---------------------------------------------------------
// Loads and stores that are coherent across the whole device while the kernel runs (the L2 caches of the chip's eight
// dies are not, for ordinary accesses): what workgroups of one launch hand to each other goes through these.
static __device__ __forceinline__ void device_store(float * p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (p: a multiple of 8 bytes)
static __device__ __forceinline__ void device_store2(float * p, float v0, float v1) {
    __hip_atomic_store((uint64_t *)p, __builtin_bit_cast(uint64_t, make_float2(v0, v1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// `bytes` bytes from `base` on as a buffer, base and length the same for every lane: loads behind its end give zeros and do not
// reach memory.  (Descriptor word 3: raw dwords.)
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t fattn_buffer(const void * base, uint32_t bytes) {
    const uint64_t b = (uint64_t)base;
    const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    return __builtin_amdgcn_make_buffer_rsrc((void *)u, 0, __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}
constexpr uint32_t FATTN_NO_ADDRESS = 0xFFFFFFF0u;          // an offset behind every buffer's end

// 16 bytes a lane from a buffer (fattn_buffer) to LDS address to + at + 16 * lane: `off` moves on by `inc` and is where they lie.  The add
// stands between the write of m0 and the load that reads it, which have to be an instruction apart.  In asm for load_to_lds16's reason.
static __device__ __forceinline__ void buffer_to_lds16(__amdgpu_buffer_rsrc_t buf, uint32_t & off, uint32_t inc, uint32_t to, uint32_t at) {
    asm volatile("s_add_i32 m0, %3, %4\n\tv_add_u32 %0, %2, %0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 : "+v"(off) : "s"(buf), "s"(inc), "s"(to), "s"(at) : "memory", "m0", "scc");
}
// the same with an offset that stays as it is
static __device__ __forceinline__ void buffer_to_lds16(__amdgpu_buffer_rsrc_t buf, uint32_t off, uint32_t to, uint32_t at) {
    asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(buf), "s"(to), "s"(at) : "memory", "m0", "scc");
}
// the same with 4 bytes a lane
static __device__ __forceinline__ void buffer_to_lds4(__amdgpu_buffer_rsrc_t buf, uint32_t & off, uint32_t inc, uint32_t to, uint32_t at) {
    asm volatile("s_add_i32 m0, %3, %4\n\tv_add_u32 %0, %2, %0\n\tbuffer_load_dword %0, %1, 0 offen lds"
                 : "+v"(off) : "s"(buf), "s"(inc), "s"(to), "s"(at) : "memory", "m0", "scc");
}

// out[row] = sum_s acc_s * exp(m_s - M) / sum_s l_s * exp(m_s - M), for the four values d4*4 .. d4*4+3 of the row, folded in in
// split order.  DEVICE: the partials come from other workgroups of this launch (and the rows of a wave rise with its lanes, all
// their partials within 4 GiB).
// The (m, l) pairs and the accumulators of 4, 8 or 16 splits are requested together, so that a row costs one memory round trip
// up to 16 splits.  What counts beside that round trip is the number of requests: they take 16 bytes (two pairs, or four values)
// and ask memory for nothing behind the last split.  Against batches of 8 in 8-byte requests, the next batch behind a branch
// (for which the compiler waited as if for both), with the counters below, us a call inside a graph: 5 rows x 20 heads of 64,
// 8 splits 7.83 -> 7.0; 8 heads of 128, 7 splits of Q8_0 7.8 -> 7.45, 13 splits of f16 9.9 -> 9.1, 16 of Q4_0 9.9 -> 8.8.  More than 16 splits
// are batches of 16 one after another, without the next one ahead: 8 heads of 128 against 8192 keys in 32 splits 15.2 -> 11.85, in 64 20.8 ->
// 14.55.  In a launch of its own, whose requests past the end are not free, up to 8 that are left over are a batch of 8: the tile kernel's
// 22 ranges of 64 x 4 heads 12.3 in batches of 8, 12.65 in two of 16, 12.2 like this; 32 ranges 12.75 -> 12.6, 64 16.5 -> 16.0.
template <bool DEVICE>
static __device__ __forceinline__ void fattn_merge_row(const FattnArgs & a, int64_t row, int d4) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const int n   = a.n_splits;
    const int lpr = a.D / 4;
    const float2 * pm = (const float2 *)(a.part_ml + (size_t)row * n * 2);
    const float4 * pa = (const float4 *)(a.part_acc + (size_t)row * n * a.D) + d4;
    float4 out = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float  M = -INFINITY, L = 0.0f;
    auto fold = [&](auto batch, int s0) __attribute__((always_inline)) {
        constexpr int NB = decltype(batch)::value;
        float2 ml[NB];
        float4 v[NB];
        if constexpr (DEVICE) {
            const int64_t  first = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(row >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)row);
            const uint64_t after = (uint64_t)((int64_t)a.Nq * a.Hq * a.B - first) * n;          // splits of the rows from there on
            const auto     bm = fattn_buffer(a.part_ml + (size_t)first * n * 2, (uint32_t)min(after * 8, (uint64_t)0xFFFFFFE0u));
            const auto     ba = fattn_buffer(a.part_acc + (size_t)first * n * a.D, (uint32_t)min(after * a.D * 4, (uint64_t)0xFFFFFFE0u));
            const uint32_t at = (uint32_t)(row - first) * (uint32_t)n;
#pragma unroll
            for (int i = 0; i < NB; i += 2) {
                const u4 x = __builtin_amdgcn_raw_buffer_load_b128(bm, (int)(s0 + i < n ? (at + s0 + i) * 8 : FATTN_NO_ADDRESS), 0, 16);      // sc1
                ml[i]     = make_float2(__uint_as_float(x[0]), __uint_as_float(x[1]));
                ml[i + 1] = make_float2(__uint_as_float(x[2]), __uint_as_float(x[3]));
            }
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const u4 x = __builtin_amdgcn_raw_buffer_load_b128(ba, (int)(s0 + i < n ? ((at + s0 + i) * lpr + d4) * 16 : FATTN_NO_ADDRESS), 0, 16);
                v[i] = make_float4(__uint_as_float(x[0]), __uint_as_float(x[1]), __uint_as_float(x[2]), __uint_as_float(x[3]));
            }
        } else {
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const int s = min(s0 + i, n - 1);           // (past the end: a second look at the last one, not used)
                ml[i] = pm[s];
                v[i]  = pa[(size_t)s * lpr];
            }
        }
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (s0 + i >= n) ml[i].x = -INFINITY;
        float Mb = M;
#pragma unroll
        for (int i = 0; i < NB; i++) Mb = fmaxf(Mb, ml[i].x);
        if (Mb == -INFINITY) return;                // nothing visible so far
        const float f = __expf(M - Mb);             // M = -inf gives 0
        L *= f; out.x *= f; out.y *= f; out.z *= f; out.w *= f;
        M = Mb;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            // a split that saw no key carries m = -inf and an accumulator that must not be touched (select, not multiply)
            const bool  seen = ml[i].x != -INFINITY;
            const float w    = seen ? __expf(ml[i].x - M) : 0.0f;
            L     += seen ? ml[i].y * w : 0.0f;
            out.x += seen ? v[i].x * w : 0.0f;
            out.y += seen ? v[i].y * w : 0.0f;
            out.z += seen ? v[i].z * w : 0.0f;
            out.w += seen ? v[i].w * w : 0.0f;
        }
    };
    if (n <= 4)      fold(std::integral_constant<int, 4>{}, 0);
    else if (n <= 8) fold(std::integral_constant<int, 8>{}, 0);
    else
        for (int s0 = 0; s0 < n; s0 += 16) {
            if (!DEVICE && n - s0 <= 8) fold(std::integral_constant<int, 8>{}, s0);
            else                        fold(std::integral_constant<int, 16>{}, s0);
        }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    out.x *= inv; out.y *= inv; out.z *= inv; out.w *= inv;
    // (dst rows are Dv floats - the head size - also where the partial rows are those of a head zero-padded to D)
    if (d4 * 4 < a.Dv) *((float4 *)(a.dst + (size_t)row * a.Dv) + d4) = out;
}

// The end of a workgroup that has stored its partials, when the launch merges in the kernel (a.counters): true for the
// one workgroup of set `group` that finds the other n - 1 done.  The partials were stored by device_store (a thread that
// used ordinary stores says so with `wrote_plain`, and pays for a write-back of its die's whole L2): every thread waits
// for its stores to be acknowledged before the workgroup counts itself done, and the merging workgroup reads by
// device_load.  All threads of the workgroup must call this; `flag` is a word of LDS that nothing else uses from here on.
// The counter wraps to zero when the set is complete.
// The sets' counters lie on cache lines of their own: the chip performs atomics on one line one after another.  Workgroups that
// only store, count and leave, all at the same time: 8 sets of 7 splits 2.7 us a launch with the counters side by side and a
// store that clears them, 2.0 like this; 20 of 8 3.6, 2.1; 8 of 16 3.4, 2.1 (an empty launch 1.65).
constexpr int FATTN_COUNTERS = 16384;              // a set number's own line below 512, shared by 32 at most beyond
static __device__ __forceinline__ uint32_t fattn_counter_of(int64_t group) {
    constexpr uint32_t LINE = 32, LINES = FATTN_COUNTERS / LINE;
    return (uint32_t)group % LINES * LINE + (uint32_t)group / LINES;
}
static __device__ __forceinline__ bool fattn_last_of_set(const FattnArgs & a, int64_t group, int n, int * flag, bool wrote_plain) {
    if (wrote_plain) __threadfence();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) *flag = atomicInc(a.counters + fattn_counter_of(group), (unsigned)(n - 1)) == (unsigned)(n - 1);
    __syncthreads();
    return *flag != 0;
}

template <int GROUP>
static __device__ __forceinline__ float group_min(float x) { return -group_max<GROUP>(-x); }

// ---- block-32 storage types ------------------------------------------------------------
// BYTES per block, offsets of the quants (QS), of the fifth bits (QH, 0 = none) and whether a minimum follows the scale
template <int TYPE> struct BlockFormat;
template <> struct BlockFormat<MI355X_TYPE_Q4_0> { static constexpr int BYTES = 18, QS = 2, QH = 0, LEVELS = 16; static constexpr bool HAS_M = false; };
template <> struct BlockFormat<MI355X_TYPE_Q4_1> { static constexpr int BYTES = 20, QS = 4, QH = 0, LEVELS = 16; static constexpr bool HAS_M = true;  };
template <> struct BlockFormat<MI355X_TYPE_Q5_0> { static constexpr int BYTES = 22, QS = 6, QH = 2, LEVELS = 32; static constexpr bool HAS_M = false; };
template <> struct BlockFormat<MI355X_TYPE_Q5_1> { static constexpr int BYTES = 24, QS = 8, QH = 4, LEVELS = 32; static constexpr bool HAS_M = true;  };
template <> struct BlockFormat<MI355X_TYPE_Q8_0> { static constexpr int BYTES = 34, QS = 2, QH = 0, LEVELS = 256; static constexpr bool HAS_M = false; };

static inline __host__ __device__ int fattn_block_bytes(int type) {
    switch (type) {
        case MI355X_TYPE_Q4_0: return 18;
        case MI355X_TYPE_Q4_1: return 20;
        case MI355X_TYPE_Q5_0: return 22;
        case MI355X_TYPE_Q5_1: return 24;
        case MI355X_TYPE_Q8_0: return 34;
        default:               return 0;
    }
}

// elements j0 .. j0+N-1 (N = 4 or 8, j0 a multiple of it) of one block as f32: q*d is exact, q*d + m is one product and one
// sum, each rounded to f32 (not fused).  Blocks are only 2-byte aligned: halfword reads.
template <int TYPE, int N>
static __device__ __forceinline__ void dequant(const char * blk, int j0, float (&out)[N]) {
    typedef BlockFormat<TYPE> F;
    const float d = h2f_bits(*(const uint16_t *)blk);
    if (TYPE == MI355X_TYPE_Q8_0) {
        const uint16_t * qs = (const uint16_t *)(blk + 2 + j0);
#pragma unroll
        for (int i = 0; i < N / 2; i++) {
            const uint16_t w = qs[i];
            out[2 * i]     = (float)(int8_t)(w & 0xff) * d;
            out[2 * i + 1] = (float)(int8_t)(w >> 8) * d;
        }
        return;
    }
    const float m = F::HAS_M ? h2f_bits(*(const uint16_t *)(blk + 2)) : 0.0f;
    const uint16_t * qs = (const uint16_t *)(blk + F::QS + (j0 & 15));      // elements j and j + 16 share a byte
    const int sh = (j0 & 16) ? 4 : 0;
    uint32_t hb = 0;
    if (F::QH) {
        const uint16_t * qh = (const uint16_t *)(blk + F::QH);
        hb = (((uint32_t)qh[0] | (uint32_t)qh[1] << 16) >> j0) & 0xffu;
    }
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
        const uint32_t w  = qs[i];
        const int      q0 = (int)(((w >> sh) & 15u) | (((hb >> (2 * i)) & 1u) << 4));
        const int      q1 = (int)(((w >> (8 + sh)) & 15u) | (((hb >> (2 * i + 1)) & 1u) << 4));
        if (F::HAS_M) {
            out[2 * i]     = mul_then_add((float)q0, d, m);
            out[2 * i + 1] = mul_then_add((float)q1, d, m);
        } else {
            out[2 * i]     = (float)(q0 - F::LEVELS / 2) * d;
            out[2 * i + 1] = (float)(q1 - F::LEVELS / 2) * d;
        }
    }
}

// One CPY / SET_ROWS node.
struct CpyArgs {
    const char * src;
    char *       dst;
    int64_t sne[4], dne[4];
    int64_t snb[4], dnb[4];
    FastDiv sdiv[3], ddiv[3];  // of the launch's units: units along dimension 0, extents of dimensions 1 and 2 (filled in by the launcher)
    int32_t same_shape;        // sne == dne (likewise)
    int64_t n;                 // elements (or blocks of 32 when a side is a block type)
    int64_t mirror;            // 0, or the distance in bytes from dst to a second copy that gets the same stores
    int32_t whole;             // what the destination is whole pieces of: 128-byte lines 2, 32-byte sectors 1, else 0 (filled in by the launcher)
    // SET_ROWS only
    const char * idx;
    int32_t idx_is_i64;
    int64_t ine[3], inb[3];
};

// The relative-position mask of a FastConformer attention block (relpos.hip).
struct RelposArgs {
    const char * qv;  size_t nbq1, nbq2, nbq3;                  // F32 [D, Nq, H, B]
    const char * r;   size_t nbr1, nbr2, nbr3; int32_t Hr, Br;   // F32 | F16 [D, Nq+Nkv-1, Hr, Br]
    const char * add; size_t nba1, nba2, nba3; int32_t Ha, Ba;   // optional F32 | F16 [>=Nkv, >=Nq, Ha, Ba]
    int32_t add_f16;
    char *       out; size_t nbo1, nbo2, nbo3;                  // F16 [Nkv, Nq, H, B], rows contiguous
    int32_t out_al4;                                            // out base and strides are multiples of 4 bytes
    int32_t D, Nq, Nkv, H, B;
    float   scale;
    int32_t n_cus;                                              // CUs of the device (0 = unknown)
    int32_t n_qblocks, n_chunks, chunk_tiles;                   // filled in by the launcher
};

// FastConformer's relative-position attention in one kernel (fattn_relpos.hip): K, V and the table are f16
struct FattnRelposArgs {
    const char * qu;  int64_t nbu1, nbu2, nbu3;                  // F32 [D, Nq, H, B]: q + pos_bias_u
    const char * qv;  int64_t nbw1, nbw2, nbw3;                  // F32 [D, Nq, H, B]: q + pos_bias_v
    const char * k;   int64_t nbk1, nbk2, nbk3;                  // F16 [D, Nkv, H / gqa, B / bq]
    const char * v;   int64_t nbv1, nbv2, nbv3;
    const char * r;   int64_t nbr1, nbr2, nbr3; int32_t Hr, Br;   // F16 [D, Nq+Nkv-1, Hr, Br]
    const char * add; int64_t nba1, nba2, nba3; int32_t Ha, Ba;   // optional F32 | F16 [>=Nkv, >=Nq, Ha, Ba]
    int32_t add_f16;
    float *      dst;                                            // F32 [D, H, Nq, B] contiguous
    int32_t D, Nq, Nkv, H, B, gqa, bq;
    int32_t n_cus;
    float   scale;
};

// Launchers implemented next to their kernels; all return hipError_t as int.
int fattn_vec_launch(const FattnArgs & a, int ktype, hipStream_t stream);
int fattn_vec_form(const FattnArgs & a, int ktype);              // mi355x_fattn_form of the call, as its launcher decides it
int fattn_merge_launch(const FattnArgs & a, hipStream_t stream);
int fattn_mma_launch(const FattnArgs & a, int ktype, hipStream_t stream);
// the instantiation of the tile kernel a call takes
struct FattnMmaVariant {
    int  query_blocks;            // 32-query blocks per wave (1 or 2)
    int  key_split;               // 2: the waves of a workgroup pair up over the two halves of every key tile
    int  queries_per_workgroup;   // of four waves
    bool direct;                  // K/V tiles move global -> LDS without passing registers
    bool mask_dma;                // so does the mask
};
void fattn_mma_variant(const FattnArgs & a, int ktype, FattnMmaVariant & v);
// waves of a workgroup of the pipelined kernel, which takes the variant's place, or 0: the tile kernel's (four)
int fattn_pipe_waves(const FattnArgs & a, int ktype, const FattnMmaVariant & v);
bool fattn_pipe_reaches(const FattnArgs & a, int64_t keys, bool shared_q);   // a range of so many keys, its waves sharing their queries or not
bool fattn_pipe_alone(const FattnArgs & a, const FattnMmaVariant & v);       // (of its calls) waves that take different keys of the same queries
int fattn_pipe_launch(const FattnArgs & a, const FattnMmaVariant & v, int waves, hipStream_t stream);
bool fattn_mma_supported(const FattnArgs & a, int ktype);
int fattn_decode_launch(const FattnArgs & a, int ktype, hipStream_t stream);
int fattn_decode_form(const FattnArgs & a, int ktype);
bool fattn_decode_supported(const FattnArgs & a, int ktype);
int cpy_launch(const CpyArgs & a, int stype, int dtype, hipStream_t stream);
int set_rows_launch(const CpyArgs & a, int dtype, hipStream_t stream);
int fill_launch(void * ptr, int value, size_t size, hipStream_t stream);      // memset by a kernel
int relpos_bias_launch(RelposArgs a, int rtype, hipStream_t stream);
int fattn_relpos_launch(const FattnRelposArgs & a, hipStream_t stream);
bool fattn_relpos_supported(const FattnRelposArgs & a);
// an F32 tensor [D, ne1, ne2, ne3] (D = the attention call's head size, rows 16-byte aligned) converted to a contiguous f16
// copy by the same launch; n = its 8-element chunks
// (kv_to_f16_launch: K and V, of any storage type each and any strides, -> contiguous f16 [D, Nkv, Hkv, Bk] at dst and right
//  behind it; the rider only beside a K and V of one type)
struct F32Rider {
    const char * src;
    char *       dst;
    int64_t ne1, ne2, nb1, nb2, nb3, n;
};
int kv_to_f16_launch(const FattnArgs & a, int ktype, int vtype, void * dst, hipStream_t stream, const F32Rider * rider = nullptr);
