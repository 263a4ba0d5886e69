// GGML_OP_CPY / CONT / DUP / SET_ROWS with the destination in device memory: the KV-cache
// writes that feed FLASH_ATTN_EXT (src/crispasr.cpp:2810-2811, 3185-3203, 2956-2973;
// src/core/attention.h:342-378) and the dequantising reads (src/core/attention.h:917-920).
// HBM-bound byte work, 8 elements per lane wherever rows allow it, coalesced along dimension 0.  Source and destination may have different shapes with equal element
// counts (the reference copies a [n_state, n_ctx] tensor into a 1-D cache view).
#include "copy_forms.h"

#include <string.h>
#include <type_traits>

// The quantisers must round every product and every sum on its own, as the reference's scalar code does: hipcc's default
// contraction turns x * id + c into one fused multiply-add (so do __fmul_rn / __fadd_rn, which inline as contractible), and
// an element whose sum lands within half an ulp of an integer then truncates to the neighbouring level.
#pragma clang fp contract(off)

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

// Which element a thread works on: unit i of `unit0` elements each -> its place along the four dimensions.
// I = uint32_t (up to 2^31 units): divisions by multiply and shift, four instructions each.  In 64-bit arithmetic the six
// divisions of a copy are loops of a hundred instructions each and most of a small launch's time (the 5 x 1280 values of a
// decoder step into their F16 cache: 2.87 us with them, 1.92 without; a token's rows into a Q8_0 cache 2.94 -> 1.96; a
// dequantising read of 663 x 8 rows of 128 4.8 -> 3.2: the shortest launch takes about 1.3).
struct Place {
    int64_t i0, i1, i2, i3;                 // i0 in units
};
template <typename I>
__device__ __forceinline__ Place place_of(I i, const int64_t (&ne)[4], const FastDiv (&div)[3], int64_t unit0) {
    Place p;
    if constexpr (sizeof(I) == 4) {
        const uint32_t r1 = divide(i, div[0]), r2 = divide(r1, div[1]), r3 = divide(r2, div[2]);
        p.i0 = i - r1 * div[0].d;
        p.i1 = r1 - r2 * div[1].d;
        p.i2 = r2 - r3 * div[2].d;
        p.i3 = r3;
    } else {
        const int64_t n0 = ne[0] / unit0;
        p.i0 = i % n0;    i /= n0;
        p.i1 = i % ne[1]; i /= ne[1];
        p.i2 = i % ne[2];
        p.i3 = i / ne[2];
    }
    return p;
}
// its byte offset; step0 = bytes from one unit to the next along dimension 0
__device__ __forceinline__ int64_t offset_at(const Place & p, const int64_t (&nb)[4], int64_t step0) {
    return p.i0 * step0 + p.i1 * nb[1] + p.i2 * nb[2] + p.i3 * nb[3];
}
template <typename I> __device__ __forceinline__ I thread_index() { return (I)blockIdx.x * 256 + threadIdx.x; }
// Lanes of the grid, by which the kernels that give a lane four elements of 64-bit indices walk on: a grid has fewer than 2^32.
template <typename I> __device__ __forceinline__ I grid_lanes() { return (I)gridDim.x * 256; }
constexpr int64_t MAX_WALKED = (int64_t)1 << 31;

// the wide form of a copy or SET_ROWS: everything the narrow one does not hold
template <typename I> struct WideCopy : CpyArgs {
    typedef I       index;
    typedef int64_t offset;
};
template <typename I>
__device__ __forceinline__ void offsets(const WideCopy<I> & a, I i, int unit0, int64_t sstep, int64_t dstep, int64_t & so, int64_t & to) {
    const Place s = place_of<I>(i, a.sne, a.sdiv, unit0);
    Place d = s;
    if (!a.same_shape) d = place_of<I>(i, a.dne, a.ddiv, unit0);
    so = offset_at(s, a.snb, sstep);
    to = offset_at(d, a.dnb, dstep);
}

// bytes from one source element to the next (a destination's are always adjacent)
template <typename T> __device__ __forceinline__ int64_t element_pitch(const NarrowCopy &) { return sizeof(T); }
template <typename T, typename I> __device__ __forceinline__ int64_t element_pitch(const WideCopy<I> & a) { return a.snb[0]; }

// Sixteen bytes a lane, whole lines a wave.  Written through, they leave the dies' L2 caches while the launch still runs instead of
// at its end; marked non-temporal (STREAM) they do not stay in the memory-side cache either.  us a launch, plain / written through /
// both: F32 -> F16 rows of 128, 663 x 8 2.40 / 2.29 / 2.29, 2048 x 64 24.1 / 23.2 / 22.6; Q8_0 -> F32, 663 x 8 2.32 / 2.15 / 2.15, 2048 x 8
// 3.84 / 3.88 / 2.78, 2048 x 64 17.9 / 17.7 / 11.4.  So dequantised reads, which outgrow the caches, are both; what the next
// launch reads is written through only (six encoder layers whose K and V are copied to F16 first: 119 us plain, 118 written
// through, 124 both).  Pieces of lines written through cost up to twice the plain stores: other kernels keep plain ones, and so do
// these where the destination's rows are not whole 32-byte sectors; non-temporal ones need whole 128-byte lines.  2048 x 64 rows into a
// token-major destination, plain / written through / non-temporal as well: F16 rows of 48 bytes 3.8 / 4.6, of 80 6.7 / 7.7; F32 rows of 96
// bytes 5.7 / 4.5, of 160 7.1 / 5.3, F16 rows of 128 at 192 7.15 / 5.6; Q8_0 -> F32 rows of 512 at 544 15.0 / 13.6 / 22.1, at 512 13.0 (all).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool STREAM, typename T> __device__ __forceinline__ void store16(const NarrowCopy & a, uint32_t to, T x) {
    // (buffer stores, because only their builtin takes the cache bits: 2 = non-temporal, 16 = write through)
    const auto r = __builtin_amdgcn_make_buffer_rsrc(a.dst, 0, -1, 0x00020000);
    if (STREAM && a.whole == 2) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, (int)to, 0, 18);
    else if (a.whole)           __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, (int)to, 0, 16);
    else                        *(T *)(a.dst + to) = x;
}
template <bool STREAM, typename I, typename T> __device__ __forceinline__ void store16(const WideCopy<I> & a, int64_t to, T x) {
    if (STREAM && a.whole == 2) __builtin_nontemporal_store(x, (T *)(a.dst + to));
    else                        *(T *)(a.dst + to) = x;
}

// a kernel's arguments, taken apart where they come in the order of their loads
template <typename A> __device__ __forceinline__ const A & opened(const A & a) { return a; }
__device__ __forceinline__ NarrowCopy opened(const NarrowCopyHead & a) { return narrow_of(a); }

template <typename A, typename TS, typename TD>
__global__ void __launch_bounds__(256) cpy_scalar_kernel(const A args) {
    const auto & a = opened(args);
    typedef typename A::index I;
    const I i = thread_index<I>();
    if (i >= (I)a.n) return;
    typename A::offset so, to;
    offsets(a, i, 1, element_pitch<TS>(a), sizeof(TD), so, to);
    const TS x = *(const TS *)(a.src + so);
    char * dp = a.dst + to;
    *(TD *)dp = (TD)x;                                          // f32 -> f16 is round-to-nearest-even
    if (a.mirror) *(TD *)(dp + a.mirror) = (TD)x;
}

typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

// What a lane's 16-byte store of TD holds, 8 or 4 consecutive elements of dimension 0, for f16 <-> f32 and same-type copies.
// Launched only when dimension 0 is whole such units on both sides, the elements are adjacent and rows start on the 16 bytes
// (8 where four f16 are read) that a lane moves at once.
template <typename TD> constexpr int vec_elements() { return 16 / (int)sizeof(TD); }
template <typename TS, typename TD, typename A>
__device__ __forceinline__ void cpy_vec_body(const A & a) {
    typedef typename A::index I;
    constexpr int E = vec_elements<TD>();
    constexpr int SAL = E * (int)sizeof(TS) < 16 ? E * (int)sizeof(TS) : 16;
    typedef TS Src __attribute__((ext_vector_type(E), aligned(SAL)));
    typedef TD Dst __attribute__((ext_vector_type(E)));
    for (I i = thread_index<I>(); i < (I)a.n; i += grid_lanes<I>()) {
        typename A::offset so, to;
        offsets(a, i, E, E * sizeof(TS), E * sizeof(TD), so, to);
        const Src x = *(const Src *)(a.src + so);
        Dst y;
#pragma unroll
        for (int e = 0; e < E; e++) y[e] = (TD)x[e];
        store16<false>(a, to, y);
        if (a.mirror) *(Dst *)(a.dst + to + a.mirror) = y;
        if (sizeof(I) == 4) return;
    }
}
template <typename A, typename TS, typename TD>
__global__ void __launch_bounds__(256) cpy_vec_kernel(const A args) { cpy_vec_body<TS, TD>(opened(args)); }
template <typename TS, typename TD>
__global__ void __launch_bounds__(256) cpy_vec_kernel_head(FATTN_HEAD_PARAMS, const ArgTail<NarrowCopyHead> tail) {
    cpy_vec_body<TS, TD>(narrow_of(fattn_join<NarrowCopyHead>(FATTN_HEAD_ARGS, tail)));
}

// Quantise one block of 32 held by a quad of lanes, 8 consecutive elements each (lane c of the quad: elements 8c .. 8c+7),
// and store it.  Called by all four lanes: the quad's reductions are two DPP steps, and a lane stores 8 bytes of
// quants at once.  Against one element per lane, 32 lanes per block and a byte store each: 1 GiB of F32 into Q8_0
// 1678 -> 275 us (4.9 TB/s, the rate of a plain copy), the 407 x 8 rows of a prompt 5.2 -> 3.3 us.
//   Q8_0: d = amax/127 (f32), q = rne(x * (1/d)), d stored as fp16
//   Q4_0 / Q5_0: d = (signed value of largest magnitude, the first one) / -8 (-16), q = min(15 (31), trunc(x/d + 8.5 (16.5)))
//   Q4_1 / Q5_1: d = (max - min) / 15 (31), m = min, q = min(15 (31), trunc((x - min)/d + 0.5))
// every product and sum is a single f32 operation, none fused.
// mirror: 0, or the distance to a second copy of the destination that gets the same bytes
template <int TYPE>
__device__ __forceinline__ void quantize_block_store(const float (&x)[8], char * blk, int c, bool ok, int64_t mirror) {
    typedef BlockFormat<TYPE> F;
    const int copies = mirror ? 2 : 1;
    if (TYPE == MI355X_TYPE_Q8_0) {
        float amax = fabsf(x[0]);
#pragma unroll
        for (int e = 1; e < 8; e++) amax = fmaxf(amax, fabsf(x[e]));
        amax = group_max<4>(amax);
        const float d  = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        u32x2_a2 q = {0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; e++) q[e >> 2] |= ((uint32_t)(int)rintf(x[e] * id) & 0xFFu) << (8 * (e & 3));
        if (ok) {
            for (int k = 0; k < copies; k++, blk += mirror) {
                *(u32x2_a2 *)(blk + 2 + c * 8) = q;
                if (c == 0) *(_Float16 *)blk = (_Float16)d;
            }
        }
        return;
    }
    float d, m = 0.0f;
    uint32_t q[8];
    if (!F::HAS_M) {
        // the first element of largest magnitude, with its sign: within the lane, then the lowest lane that has it
        float ext = x[0], amax = fabsf(x[0]);
#pragma unroll
        for (int e = 1; e < 8; e++) {
            if (fabsf(x[e]) > amax || amax != amax) {
                amax = fabsf(x[e]);
                ext  = x[e];
            }
        }
        const float top = group_max<4>(amax);
        float first = 0.0f;
#pragma unroll
        for (int k = 3; k >= 0; k--) {
            const float a = quad_broadcast(amax, k), v = quad_broadcast(ext, k);
            if (a == top) first = v;
        }
        d = (top > 0.0f ? first : 0.0f) / (float)(-(F::LEVELS / 2));
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x0 = x[e] * id;
            const int   qi = (int)(int8_t)(int)(x0 + ((float)(F::LEVELS / 2) + 0.5f));
            q[e] = (uint32_t)(qi < F::LEVELS - 1 ? qi : F::LEVELS - 1);
        }
    } else {
        float lo = -x[0], hi = x[0];
#pragma unroll
        for (int e = 1; e < 8; e++) {
            lo = fmaxf(lo, -x[e]);
            hi = fmaxf(hi, x[e]);
        }
        m = -group_max<4>(lo);
        d = (group_max<4>(hi) - m) / (float)(F::LEVELS - 1);
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x0 = (x[e] - m) * id;
            const int   qi = (int)(uint8_t)(int)(x0 + 0.5f);
            q[e] = (uint32_t)(qi < F::LEVELS - 1 ? qi : F::LEVELS - 1);
        }
    }
    // elements j and j + 16 share a byte: lanes 0 and 1 take the low nibbles from themselves, the high ones from lanes 2 and 3
    u32x2_a2 lo = {0u, 0u}, by;
    uint32_t bits = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        lo[e >> 2] |= (q[e] & 15u) << (8 * (e & 3));
        bits |= ((q[e] >> 4) & 1u) << e;
    }
#pragma unroll
    for (int k = 0; k < 2; k++) by[k] = lo[k] | quad_swap2(lo[k]) << 4;
    uint32_t qh = bits << (8 * c);                       // the fifth bits of the whole block in every lane
    qh |= quad_swap1(qh);
    qh |= quad_swap2(qh);
    if (ok) {
        for (int k = 0; k < copies; k++, blk += mirror) {
            if (c < 2) *(u32x2_a2 *)(blk + F::QS + 8 * c) = by;
            if (c == 2) {
                *(_Float16 *)blk = (_Float16)d;
                if (F::HAS_M) *(_Float16 *)(blk + 2) = (_Float16)m;
            }
            if (F::QH && c == 3) {
                *(uint16_t *)(blk + F::QH) = (uint16_t)qh;
                *(uint16_t *)(blk + F::QH + 2) = (uint16_t)(qh >> 16);
            }
        }
    }
}

// the 8 elements of a quad's lane: two 16-byte loads where the source's rows allow it
template <bool VEC>
__device__ __forceinline__ void load8(const char * p, int64_t nb0, float (&x)[8]) {
    if (VEC) {
        const float4v u = *(const float4v *)p, v = *(const float4v *)(p + 16);
#pragma unroll
        for (int e = 0; e < 4; e++) { x[e] = u[e]; x[4 + e] = v[e]; }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = *(const float *)(p + e * nb0);
    }
}

// F32 -> block type; one block per 4 lanes
template <typename A, int TYPE, bool VEC>
__global__ void __launch_bounds__(256) cpy_f32_block_kernel(const A a) {
    typedef typename A::index I;
    const I    blk = (I)blockIdx.x * 64 + (threadIdx.x >> 2);
    const int  c   = threadIdx.x & 3;
    const bool ok  = blk < (I)a.n;
    const int64_t es = VEC ? 4 : element_pitch<float>(a);              // bytes from one F32 element to the next
    typename A::offset so, to;
    offsets(a, ok ? blk : 0, FATTN_QK8_0, FATTN_QK8_0 * es, BlockFormat<TYPE>::BYTES, so, to);
    float x[8];
    load8<VEC>(a.src + so + c * 8 * es, es, x);
    quantize_block_store<TYPE>(x, a.dst + to, c, ok, a.mirror);
}

// block type -> F32; 4 elements per lane, eight lanes per block, so that with 16-byte stores (VEC) a wave writes 1 KB that lies
// together: with 8 elements, two stores and half as many lanes 663 x 8 rows of 128 took 2.51 us instead of 2.15, 2048 x 64 20.6 instead of 11.4.
template <typename A, int TYPE, bool VEC>
__global__ void __launch_bounds__(256) cpy_block_f32_kernel(const A args) {
    const auto & a = opened(args);
    typedef typename A::index I;
    const int j0  = (threadIdx.x & 7) * 4;
    for (I blk = (I)blockIdx.x * 32 + (threadIdx.x >> 3); blk < (I)a.n; blk += grid_lanes<I>() / 8) {
        typename A::offset so, to;
        offsets(a, blk, FATTN_QK8_0, BlockFormat<TYPE>::BYTES, FATTN_QK8_0 * 4, so, to);
        float y[4];
        dequant<TYPE>(a.src + so, j0, y);
        if (VEC) {
            const float4v v = {y[0], y[1], y[2], y[3]};
            store16<true>(a, to + j0 * 4, v);
            if (a.mirror) *(float4v *)(a.dst + to + j0 * 4 + a.mirror) = v;
        } else {
            char * dp = a.dst + to + j0 * 4;
            for (int k = 0; k < (a.mirror ? 2 : 1); k++, dp += a.mirror)
#pragma unroll
                for (int e = 0; e < 4; e++) ((float *)dp)[e] = y[e];
        }
        if (sizeof(I) == 4) return;
    }
}

// same block type on both sides: move the blocks as halfwords
template <typename A, int TYPE>
__global__ void __launch_bounds__(256) cpy_block_block_kernel(const A args) {
    const auto & a = opened(args);
    typedef typename A::index I;
    constexpr int HW = BlockFormat<TYPE>::BYTES / 2;
    const I   t   = thread_index<I>();
    const I   blk = t / HW;
    const int w   = (int)(t % HW);
    if (blk >= (I)a.n) return;
    typename A::offset so, to;
    offsets(a, blk, FATTN_QK8_0, BlockFormat<TYPE>::BYTES, BlockFormat<TYPE>::BYTES, so, to);
    const uint16_t x = ((const uint16_t *)(a.src + so))[w];
    char * dp = a.dst + to + 2 * w;
    *(uint16_t *)dp = x;
    if (a.mirror) *(uint16_t *)(dp + a.mirror) = x;
}

// bytes of a unit of a destination row
template <int DTYPE, int UNIT> constexpr int row_unit_bytes() {
    if constexpr (FATTN_IS_BLOCK_TYPE(DTYPE)) return BlockFormat<DTYPE>::BYTES;
    else return UNIT * (DTYPE == MI355X_TYPE_F16 ? 2 : 4);
}

struct RowPlace {
    int64_t      so, to;                   // of the source unit; of the destination's unit in row 0
    const char * ip;                       // the row's index
    int64_t      row_pitch, rows, mirror;
    bool         i64;
};
__device__ __forceinline__ RowPlace row_place(const NarrowRows & a, uint32_t i, int, int64_t sstep, int64_t dstep) {
    uint32_t so, to, xo;
    offsets(a, i, (uint32_t)sstep, (uint32_t)dstep, so, to, xo);
    return {so, to, a.idx + xo, a.dnb[0], a.rows, 0, (a.x2_is_i64 & 1) != 0};
}
template <typename I>
__device__ __forceinline__ RowPlace row_place(const WideCopy<I> & a, I i, int unit0, int64_t sstep, int64_t dstep) {
    const Place q = place_of<I>(i, a.sne, a.sdiv, unit0);
    // (a broadcast of the indices over heads and sequences is the rule: no division then)
    const int64_t x1 = a.ine[1] == 1 ? 0 : a.ine[1] == a.sne[2] ? q.i2 : q.i2 % a.ine[1];
    const int64_t x2 = a.ine[2] == 1 ? 0 : a.ine[2] == a.sne[3] ? q.i3 : q.i3 % a.ine[2];
    RowPlace p;
    p.so = offset_at(q, a.snb, sstep);
    p.to = q.i0 * dstep + q.i2 * a.dnb[2] + q.i3 * a.dnb[3];
    p.ip = a.idx + q.i1 * a.inb[0] + x1 * a.inb[1] + x2 * a.inb[2];
    p.row_pitch = a.dnb[1];
    p.rows = a.dne[1];
    p.mirror = a.mirror;
    p.i64 = a.idx_is_i64;
    return p;
}
template <typename T> __device__ __forceinline__ int64_t element_pitch(const NarrowRows &) { return sizeof(T); }

// SET_ROWS: dst[:, idx[i1, i2 % ine1, i3 % ine2], i2, i3] = convert(src[:, i1, i2, i3]), src F32
// UNIT elements of a source row per unit: 32 by a quad of lanes (block types), 8 by a lane (F16 / F32 rows that start on 16
// bytes), or 1 by a lane.  VEC: the source is read with 16-byte loads.
template <typename A, int DTYPE, int UNIT, bool VEC>
__global__ void __launch_bounds__(256) set_rows_kernel(const A a) {
    typedef typename A::index I;
    constexpr bool BLOCKS = FATTN_IS_BLOCK_TYPE(DTYPE);
    static_assert(BLOCKS ? UNIT == FATTN_QK8_0 : (UNIT == 1 || UNIT == 8), "units");
    const I    u  = BLOCKS ? (I)blockIdx.x * 64 + (threadIdx.x >> 2) : thread_index<I>();
    const int  c  = BLOCKS ? threadIdx.x & 3 : 0;
    const bool ok = u < (I)a.n;
    const int64_t es = VEC ? 4 : element_pitch<float>(a);
    const RowPlace p = row_place(a, ok ? u : 0, UNIT, UNIT * es, row_unit_bytes<DTYPE, UNIT>());
    const char * sp = a.src + p.so + c * 8 * es;
    float x[8];
    // (lanes behind the last unit read the first one: nothing here stands under a guard, so that all loads are one round trip)
    if constexpr (UNIT == 1) x[0] = *(const float *)sp;
    else                     load8<VEC>(sp, es, x);
    const int32_t lo = *(const int32_t *)p.ip, hi = *(const int32_t *)(p.ip + (p.i64 ? 4 : 0));
    const int64_t drow = (int64_t)((uint64_t)(uint32_t)(p.i64 ? hi : lo >> 31) << 32 | (uint32_t)lo);
    // A row index outside the destination writes nothing (ggml-cpu asserts 0 <= idx < ne1 instead): a stale or
    // uninitialised index tensor must not become a write outside the cache.  The lanes stay in the block's reduction.
    const bool inside = ok && drow >= 0 && drow < p.rows;
    char * dp = a.dst + p.to + (inside ? drow : 0) * p.row_pitch;
    if constexpr (BLOCKS) {
        quantize_block_store<DTYPE>(x, dp, c, inside, p.mirror);
    } else if (inside) {
        typedef typename std::conditional<DTYPE == MI355X_TYPE_F16, _Float16, float>::type TD;
        for (int k = 0; k < (p.mirror ? 2 : 1); k++, dp += p.mirror) {
            if constexpr (UNIT == 1) {
                *(TD *)dp = (TD)x[0];
            } else {
                typedef TD V8 __attribute__((ext_vector_type(8)));
                V8 y;
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = (TD)x[e];
                *(V8 *)dp = y;
            }
        }
    }
}

// K and V of one attention call -> two contiguous f16 tensors [D, Nkv, Hkv, Bk] (K first, V right behind it), one
// launch for both.  One lane per 8 elements of a row: two 128-bit loads (F32) or 8 quants and the block's scale
// (Q8_0), one 128-bit store.  Rounding is the tile kernel's own: f32 -> f16 round-to-nearest-even, q*d exact in f32
// and then rounded once.
// An F32 table [D, n1, n2, n3] with 16-byte aligned rows may ride along (the relative-position table of a FastConformer
// block, rounded for the same call): the threads behind K's and V's write its contiguous f16 copy.
// chunks of 8 elements per row, rows per head and heads per sequence of the copies, and the same of the rider's table
struct ChunkDivs {
    FastDiv kv[3], table[3];
    int64_t kv_ne[4], table_ne[4];
};
template <typename I, int TYPE>
__global__ void __launch_bounds__(256) kv_to_f16_kernel(const FattnArgs a, char * dst, const F32Rider x, const ChunkDivs v) {
    const I half = (I)((int64_t)(a.D / 8) * a.Nkv * a.Hkv * a.Bk);      // chunks per tensor
    I i = thread_index<I>();
    if (i >= 2 * half) {
        i -= 2 * half;
        if (i >= (I)x.n) return;
        const Place p = place_of<I>(i, v.table_ne, v.table, 1);
        const int   c = (int)p.i0;
        const char * row = x.src + p.i1 * x.nb1 + p.i2 * x.nb2 + p.i3 * x.nb3;
        const float4 x0 = *(const float4 *)(row + c * 32);
        const float4 x1 = *(const float4 *)(row + c * 32 + 16);
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        h8 y;
        y[0] = (_Float16)x0.x; y[1] = (_Float16)x0.y; y[2] = (_Float16)x0.z; y[3] = (_Float16)x0.w;
        y[4] = (_Float16)x1.x; y[5] = (_Float16)x1.y; y[6] = (_Float16)x1.z; y[7] = (_Float16)x1.w;
        *(h8 *)(x.dst + (int64_t)i * 16) = y;
        return;
    }
    const bool is_v = i >= half;
    if (is_v) i -= half;
    const Place p = place_of<I>(i, v.kv_ne, v.kv, 1);
    const int   c = (int)p.i0;
    const char * row = is_v ? a.v + p.i1 * a.nbv1 + p.i2 * a.nbv2 + p.i3 * a.nbv3
                            : a.k + p.i1 * a.nbk1 + p.i2 * a.nbk2 + p.i3 * a.nbk3;
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    h8 y;
    if constexpr (TYPE == MI355X_TYPE_F32) {
        const float4 x0 = *(const float4 *)(row + c * 32);
        const float4 x1 = *(const float4 *)(row + c * 32 + 16);
        y[0] = (_Float16)x0.x; y[1] = (_Float16)x0.y; y[2] = (_Float16)x0.z; y[3] = (_Float16)x0.w;
        y[4] = (_Float16)x1.x; y[5] = (_Float16)x1.y; y[6] = (_Float16)x1.z; y[7] = (_Float16)x1.w;
    } else {
        float f[8];
        dequant<TYPE>(row + (c >> 2) * fattn_block_bytes(TYPE), (c & 3) * 8, f);
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = (_Float16)f[e];
    }
    *(h8 *)(dst + (int64_t)((is_v ? half : 0) + i) * 16) = y;
}

// The same for a K and a V of different storage types (CRISPASR_KV_QUANT_K / _V, src/core/attention.h:132-137; the
// Canary decoder hands both cache views to the op as they are, src/canary.cpp:953-972): the type is looked up per
// tensor at run time.  Scalar loads: such rows are only as aligned as their type.
// It is also the launch that pads: the copies' rows are a.D elements long, the first a.Dv of them the source row's
// (a multiple of 8), zeros behind - how the tile kernel, which has forms for 64- and 128-wide heads, gets the others.
template <typename I>
__global__ void __launch_bounds__(256) kv_to_f16_mixed_kernel(const FattnArgs a, const int ktype, const int vtype, char * dst, const ChunkDivs v) {
    const I half = (I)((int64_t)(a.D / 8) * a.Nkv * a.Hkv * a.Bk);
    I i = thread_index<I>();
    if (i >= 2 * half) return;
    const bool is_v = i >= half;
    if (is_v) i -= half;
    const Place p = place_of<I>(i, v.kv_ne, v.kv, 1);
    const int   c = (int)p.i0;
    if (c * 8 >= a.Dv) {
        *(uint4 *)(dst + (int64_t)((is_v ? half : 0) + i) * 16) = uint4{0u, 0u, 0u, 0u};
        return;
    }
    const char * row = is_v ? a.v + p.i1 * a.nbv1 + p.i2 * a.nbv2 + p.i3 * a.nbv3
                            : a.k + p.i1 * a.nbk1 + p.i2 * a.nbk2 + p.i3 * a.nbk3;
    float f[8];
    const char * blk = row + (c >> 2) * fattn_block_bytes(is_v ? vtype : ktype);
    switch (is_v ? vtype : ktype) {
        case MI355X_TYPE_F32:
#pragma unroll
            for (int e = 0; e < 8; e++) f[e] = ((const float *)row)[c * 8 + e];
            break;
        case MI355X_TYPE_F16:
#pragma unroll
            for (int e = 0; e < 8; e++) f[e] = h2f_bits(((const uint16_t *)row)[c * 8 + e]);
            break;
        case MI355X_TYPE_Q8_0: dequant<MI355X_TYPE_Q8_0>(blk, (c & 3) * 8, f); break;
        case MI355X_TYPE_Q4_0: dequant<MI355X_TYPE_Q4_0>(blk, (c & 3) * 8, f); break;
        case MI355X_TYPE_Q4_1: dequant<MI355X_TYPE_Q4_1>(blk, (c & 3) * 8, f); break;
        case MI355X_TYPE_Q5_0: dequant<MI355X_TYPE_Q5_0>(blk, (c & 3) * 8, f); break;
        default:               dequant<MI355X_TYPE_Q5_1>(blk, (c & 3) * 8, f); break;
    }
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    h8 y;
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = (_Float16)f[e];
    *(h8 *)(dst + (int64_t)((is_v ? half : 0) + i) * 16) = y;
}

// memset as a kernel: a memset node recorded into a captured graph is what a fill kernel avoids.
// 16-byte stores over the aligned middle, single bytes for the (< 16-byte) head and tail.
__global__ void __launch_bounds__(256) fill_kernel(unsigned char * p, unsigned value, size_t head, size_t n16, size_t tail) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const unsigned w = value * 0x01010101u;
    if (i < n16) *(u4 *)(p + head + i * 16) = u4{w, w, w, w};
    if (i < head) p[i] = (unsigned char)value;
    if (i < tail) p[head + n16 * 16 + i] = (unsigned char)value;
}

}  // namespace

int fill_launch(void * ptr, int value, size_t size, hipStream_t stream) {
    if (size == 0) return 0;
    size_t head = (16 - (uintptr_t)ptr % 16) % 16;
    if (head > size) head = size;
    const size_t n16  = (size - head) / 16;
    const size_t tail = size - head - n16 * 16;
    const size_t threads = n16 > 16 ? n16 : 16;                    // head and tail are below 16 bytes each
    if ((threads + 255) / 256 > 0x7fffffffu) return (int)hipErrorInvalidValue;
    fattn_launch(fill_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream,
                       (unsigned char *)ptr, (unsigned)(value & 0xff), head, n16, tail);
    return (int)hipGetLastError();
}

int kv_to_f16_launch(const FattnArgs & a, int ktype, int vtype, void * dst, hipStream_t stream, const F32Rider * rider) {
    F32Rider x;
    memset(&x, 0, sizeof(x));
    if (rider) x = *rider;
    const int64_t n = 2 * (int64_t)(a.D / 8) * a.Nkv * a.Hkv * a.Bk + x.n;
    if (n == 0) return 0;
    if ((n + 255) / 256 > 0x7fffffff) return (int)hipErrorInvalidValue;
    const dim3 g((unsigned)((n + 255) / 256));
    ChunkDivs v;
    const int64_t kv_ne[4] = {a.D / 8, a.Nkv, a.Hkv, a.Bk}, table_ne[4] = {a.D / 8, x.ne1, x.ne2, 1};
    for (int i = 0; i < 4; i++) {
        v.kv_ne[i]    = kv_ne[i];
        v.table_ne[i] = table_ne[i];
        if (i < 3) {
            v.kv[i]    = fast_div((uint32_t)kv_ne[i]);
            v.table[i] = fast_div((uint32_t)table_ne[i]);
        }
    }
    const bool small = n + 256 < ((int64_t)1 << 31);             // 32-bit indices do
    if (ktype != vtype || a.Dv != a.D) {
        if (rider) return (int)hipErrorInvalidValue;
        if (small) fattn_launch(kv_to_f16_mixed_kernel<uint32_t>, g, dim3(256), 0, stream, a, ktype, vtype, (char *)dst, v);
        else       fattn_launch(kv_to_f16_mixed_kernel<int64_t>, g, dim3(256), 0, stream, a, ktype, vtype, (char *)dst, v);
        return (int)hipGetLastError();
    }
    switch (ktype) {
#define KV16(T)                                                                                                         \
    case T:                                                                                                             \
        if (small) fattn_launch((kv_to_f16_kernel<uint32_t, T>), g, dim3(256), 0, stream, a, (char *)dst, x, v);    \
        else       fattn_launch((kv_to_f16_kernel<int64_t, T>), g, dim3(256), 0, stream, a, (char *)dst, x, v);     \
        break
        KV16(MI355X_TYPE_F32);
        KV16(MI355X_TYPE_Q8_0);
        KV16(MI355X_TYPE_Q4_0);
        KV16(MI355X_TYPE_Q4_1);
        KV16(MI355X_TYPE_Q5_0);
        KV16(MI355X_TYPE_Q5_1);
#undef KV16
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

// rows of a side whose elements of `es` bytes lie `es` apart and start on multiples of `align` bytes
static bool rows_aligned(const void * p, const int64_t (&ne)[4], const int64_t (&nb)[4], int64_t es, int64_t align) {
    if (nb[0] != es || (uintptr_t)p % align) return false;
    for (int i = 1; i < 4; i++)
        if (ne[i] > 1 && nb[i] % align) return false;
    return true;
}

// f16 <-> f32 and same-type copies: whether cpy_vec_kernel takes them
template <typename TS, typename TD>
static bool vec_ok(const CpyArgs & a) {
    constexpr int E = vec_elements<TD>(), sal = E * (int)sizeof(TS) < 16 ? E * (int)sizeof(TS) : 16;
    return a.sne[0] % E == 0 && a.dne[0] % E == 0 && rows_aligned(a.src, a.sne, a.snb, sizeof(TS), sal) &&
           rows_aligned(a.dst, a.dne, a.dnb, sizeof(TD), 16) && a.mirror % 16 == 0;
}

// the wide form's divisors for units of `unit0` elements; whether 32-bit indices do (`threads` = the grid's)
static bool prepare_index(CpyArgs & a, int64_t unit0, int64_t threads) {
    a.same_shape = 1;
    for (int i = 0; i < 4; i++) a.same_shape = a.same_shape && a.sne[i] == a.dne[i];
    a.sdiv[0] = fast_div((uint32_t)(a.sne[0] / unit0));
    a.ddiv[0] = fast_div((uint32_t)(a.dne[0] / unit0));
    for (int i = 1; i < 3; i++) {
        a.sdiv[i] = fast_div((uint32_t)a.sne[i]);
        a.ddiv[i] = fast_div((uint32_t)a.dne[i]);
    }
    return threads + 256 < ((int64_t)1 << 31);
}

// a kernel of this file over `threads` lanes for units of `unit0` elements, a.n of them: in the narrow form where `narrow` filled
// it in, else in the wide one, with 32-bit indices where they do.  walked: its 64-bit form goes on from the grid's end.  pieces: of the
// wide form, whole_pieces.
#define FORM_LAUNCH(a, unit0, threads, walked, narrow, v, pieces, KERNEL, ...)                                                 \
    do {                                                                                                                  \
        const dim3 g_((unsigned)(((threads) + 255) / 256));                                                               \
        if (narrow) {                                                                                                     \
            fattn_launch((KERNEL<decltype(v), __VA_ARGS__>), g_, dim3(256), 0, stream, v);                          \
            break;                                                                                                        \
        }                                                                                                                 \
        WideCopy<uint32_t> w_;                                                                                            \
        (CpyArgs &)w_ = a;                                                                                                \
        w_.whole = (pieces);                                                                                              \
        if (prepare_index(w_, unit0, threads)) {                                                                          \
            fattn_launch((KERNEL<WideCopy<uint32_t>, __VA_ARGS__>), g_, dim3(256), 0, stream, w_);                  \
        } else {                                                                                                          \
            WideCopy<int64_t> l_;                                                                                         \
            (CpyArgs &)l_ = w_;                                                                                           \
            const dim3 lg_((unsigned)((((walked) && (threads) > MAX_WALKED ? MAX_WALKED : (threads)) + 255) / 256));      \
            fattn_launch((KERNEL<WideCopy<int64_t>, __VA_ARGS__>), lg_, dim3(256), 0, stream, l_);                  \
        }                                                                                                                 \
    } while (0)
// (es: bytes of a source element, whole blocks counted as one; order: head_first, or as_it_is for kernels that read a NarrowCopy)
static inline const NarrowCopy & as_it_is(const NarrowCopy & a) { return a; }
#define CPY_LAUNCH(a, unit0, es, sstep, dstep, threads, walked, order, KERNEL, ...)                                            \
    do {                                                                                                                  \
        NarrowCopy v_ = {};                                                                                               \
        const bool n_ = (a).snb[0] == (int64_t)(es) && narrow_copy(a, unit0, sstep, dstep, threads, v_);                  \
        auto o_ = order(v_);                                                                                              \
        FORM_LAUNCH(a, unit0, threads, walked, n_, o_, whole_pieces((a).dst, walk_of((a).dne, (a).dnb, unit0, dstep), dstep), KERNEL, __VA_ARGS__); \
    } while (0)
#define ROWS_LAUNCH(a, unit0, threads, ...)                                                                               \
    do {                                                                                                                  \
        NarrowRows v_;                                                                                                    \
        const bool n_ = narrow_rows(a, unit0, threads, v_);                                                               \
        FORM_LAUNCH(a, unit0, threads, false, n_, v_, 0, set_rows_kernel, __VA_ARGS__);                               \
    } while (0)

template <typename TS, typename TD>
static void launch_plain(const CpyArgs & a, hipStream_t stream) {
    if (vec_ok<TS, TD>(a)) {
        constexpr int E = vec_elements<TD>();
        CpyArgs b = a;
        b.n = a.n / E;
        // More than 64 Ki lanes: the head of the arguments in registers.  Six encoder layers with twelve copies of 1500 x 512 96.3 -> 93.0 us;
        // a launch of a few workgroups ends no sooner, and one of eight numbers costs the host and, in a graph, the device 0.1 us more
        // (5 x 512 values 1.68 and 1.84 us; row writes and dequantising reads, of which steps are full, stay with the structure).
        NarrowCopy v;
        if (b.n > 65536 && b.snb[0] == (int64_t)sizeof(TS) && narrow_copy(b, E, E * sizeof(TS), E * sizeof(TD), b.n, v))
            fattn_launch_head(cpy_vec_kernel_head<TS, TD>, dim3((unsigned)((b.n + 255) / 256)), dim3(256), 0, stream, head_first(v));
        else
            CPY_LAUNCH(b, E, sizeof(TS), E * sizeof(TS), E * sizeof(TD), b.n, true, head_first, cpy_vec_kernel, TS, TD);
    } else {
        CPY_LAUNCH(a, 1, sizeof(TS), sizeof(TS), sizeof(TD), a.n, false, head_first, cpy_scalar_kernel, TS, TD);
    }
}

template <int T>
static void launch_to_blocks(const CpyArgs & a, hipStream_t stream) {
    constexpr int U = FATTN_QK8_0, BB = BlockFormat<T>::BYTES;
    if (rows_aligned(a.src, a.sne, a.snb, 4, 16)) CPY_LAUNCH(a, U, 4, U * 4, BB, a.n * 4, false, as_it_is, cpy_f32_block_kernel, T, true);
    else                                          CPY_LAUNCH(a, U, 4, U * 4, BB, a.n * 4, false, as_it_is, cpy_f32_block_kernel, T, false);
}

template <int T>
static void launch_from_blocks(const CpyArgs & a, hipStream_t stream) {
    constexpr int U = FATTN_QK8_0, BB = BlockFormat<T>::BYTES;
    if (rows_aligned(a.dst, a.dne, a.dnb, 4, 16) && a.mirror % 16 == 0) CPY_LAUNCH(a, U, BB, BB, U * 4, a.n * 8, true, head_first, cpy_block_f32_kernel, T, true);
    else                                                                CPY_LAUNCH(a, U, BB, BB, U * 4, a.n * 8, true, head_first, cpy_block_f32_kernel, T, false);
}

template <int T>
static void launch_blocks(const CpyArgs & a, hipStream_t stream) {
    constexpr int U = FATTN_QK8_0, BB = BlockFormat<T>::BYTES;
    CPY_LAUNCH(a, U, BB, BB, BB, a.n * (BB / 2), false, head_first, cpy_block_block_kernel, T);
}

int cpy_launch(const CpyArgs & a, int stype, int dtype, hipStream_t stream) {
    if (a.n == 0) return 0;
    if (stype == MI355X_TYPE_F32 && dtype == MI355X_TYPE_F32)      launch_plain<float, float>(a, stream);
    else if (stype == MI355X_TYPE_F32 && dtype == MI355X_TYPE_F16) launch_plain<float, _Float16>(a, stream);
    else if (stype == MI355X_TYPE_F16 && dtype == MI355X_TYPE_F16) launch_plain<_Float16, _Float16>(a, stream);
    else if (stype == MI355X_TYPE_F16 && dtype == MI355X_TYPE_F32) launch_plain<_Float16, float>(a, stream);
#define BLOCK_CASES(T)                                                                                                    \
    else if (stype == MI355X_TYPE_F32 && dtype == T) launch_to_blocks<T>(a, stream);                                       \
    else if (stype == T && dtype == MI355X_TYPE_F32) launch_from_blocks<T>(a, stream);                                     \
    else if (stype == T && dtype == T) launch_blocks<T>(a, stream);
    BLOCK_CASES(MI355X_TYPE_Q8_0)
    BLOCK_CASES(MI355X_TYPE_Q4_0)
    BLOCK_CASES(MI355X_TYPE_Q4_1)
    BLOCK_CASES(MI355X_TYPE_Q5_0)
    BLOCK_CASES(MI355X_TYPE_Q5_1)
#undef BLOCK_CASES
    else
        return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
}

template <int T>
static void launch_set_rows(const CpyArgs & a, hipStream_t stream) {
    const bool vec = rows_aligned(a.src, a.sne, a.snb, 4, 16);
    if constexpr (FATTN_IS_BLOCK_TYPE(T)) {
        if (vec) ROWS_LAUNCH(a, FATTN_QK8_0, a.n * 4, T, FATTN_QK8_0, true);
        else     ROWS_LAUNCH(a, FATTN_QK8_0, a.n * 4, T, FATTN_QK8_0, false);
    } else {
        const int64_t ds = T == MI355X_TYPE_F16 ? 2 : 4;
        if (vec && a.sne[0] % 8 == 0 && rows_aligned(a.dst, a.dne, a.dnb, ds, 8 * ds) && a.mirror % (8 * ds) == 0) {
            CpyArgs b = a;
            b.n = a.n / 8;
            ROWS_LAUNCH(b, 8, b.n, T, 8, true);
        } else {
            ROWS_LAUNCH(a, 1, a.n, T, 1, false);
        }
    }
}

int set_rows_launch(const CpyArgs & a, int dtype, hipStream_t stream) {
    if (a.n == 0) return 0;
    if (a.n > ((int64_t)1 << 38)) return (int)hipErrorInvalidValue;
    switch (dtype) {
        case MI355X_TYPE_Q8_0: launch_set_rows<MI355X_TYPE_Q8_0>(a, stream); break;
        case MI355X_TYPE_Q4_0: launch_set_rows<MI355X_TYPE_Q4_0>(a, stream); break;
        case MI355X_TYPE_Q4_1: launch_set_rows<MI355X_TYPE_Q4_1>(a, stream); break;
        case MI355X_TYPE_Q5_0: launch_set_rows<MI355X_TYPE_Q5_0>(a, stream); break;
        case MI355X_TYPE_Q5_1: launch_set_rows<MI355X_TYPE_Q5_1>(a, stream); break;
        case MI355X_TYPE_F16:  launch_set_rows<MI355X_TYPE_F16>(a, stream); break;
        case MI355X_TYPE_F32:  launch_set_rows<MI355X_TYPE_F32>(a, stream); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}
