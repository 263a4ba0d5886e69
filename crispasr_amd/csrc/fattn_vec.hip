// Split-KV vector attention kernel for gfx950 (wave64) and the merge of its partials.
//
// One workgroup (4 waves) owns one query row (query, head, batch) and one KV split.
// A row of K or V is spread over LPR lanes, 8 elements (one 128-bit load for f16) per
// lane, so a wave reads 64/LPR whole rows per load instruction - contiguous 128- or
// 256-byte segments.  Each group of LPR lanes keeps its own online-softmax state
// (m, l, acc[8] per lane) over the keys it visits; the dot products are reduced across
// the group with DPP butterflies.  Groups are merged with cross-lane shuffles, waves
// through LDS, and splits by fattn_merge_kernel.
//
// Semantics follow GGML_OP_FLASH_ATTN_EXT as the reference's call sites use it
// (src/crispasr.cpp:3208-3222, 3269-3282; src/core/attention.h:992; src/canary.cpp:966-972):
// s = scale*<q,k> [soft-capped] + slope*mask, -inf mask entries exclude a key, GQA by
// h / (Hq/Hkv), mask broadcast by h % Hm and b % Bm, output [D, Hq, Nq, B].
#include "fattn_row.h"

#include <stddef.h>

namespace {

constexpr int VEC_WAVES   = 4;
constexpr int VEC_THREADS = VEC_WAVES * 64;

// One (row, range) by a workgroup: row (iq1, h, b) of the result, range `split` of the keys.
// mask_of: makes the row's mask once q has been asked for (its divisions and the slope's branch ahead of q are 0.1 to 0.5 us of a call of few
// keys and 1% of a long one: 11 rows x 20 heads of 256 x 2 against 37 11.0 and 10.55 us, 25 x 4 against 25 6.35 and 6.1, 988 x 8 678 and 671).
template <int TYPE, int LPR, int PIECES, typename MaskFn, typename RequestedFn>
__device__ __forceinline__ void vec_body(const FattnArgs & a, int split, int row, const char * qbase, const char * kbase, const char * vbase,
                                         const MaskFn & mask_of, const RequestedFn & requested) {
    const int tid  = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int d0   = (lane % LPR) * 8;          // the lane's 8 elements of d (D is a multiple of 4: the last lane may hold 4)

    const int k_begin = split * a.keys_per_split;
    const int k_end   = min(a.Nkv, k_begin + a.keys_per_split);

    float q[8];
    if constexpr (PIECES > 0) {                  // 16-byte aligned rows, as a buffer that ends with the head: zeros behind it, and no wait here
        typedef float float4v __attribute__((ext_vector_type(4)));
        const __amdgpu_buffer_rsrc_t qrow = fattn_buffer(qbase, (uint32_t)a.D * 4);
        const float4v x = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(qrow, d0 * 4, 0, 0));
        const float4v y = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(qrow, d0 * 4 + 16, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            q[e]     = x[e];
            q[4 + e] = y[e];
        }
    } else {
        const float * qrow = (const float *)qbase;
#pragma unroll
        for (int e = 0; e < 8; e++) q[e] = d0 + e < a.D ? qrow[d0 + e] : 0.0f;
    }
    const RowMaskTensor mask = mask_of();

    RowPartial st;
    st.m = -INFINITY;
    st.l = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) st.acc[e] = 0.0f;
    row_scan<TYPE, TYPE, LPR, VEC_WAVES, PIECES>(row_scan_args(a), q, kbase, vbase, mask, k_begin, k_end, wave, lane, st, requested);

    // merge the waves through LDS
    __shared__ float sh[VEC_WAVES][LPR][10];
    if (lane < LPR) {
        sh[wave][lane][0] = st.m;
        sh[wave][lane][1] = st.l;
#pragma unroll
        for (int e = 0; e < 8; e++) sh[wave][lane][2 + e] = st.acc[e];
    }
    __syncthreads();
    if (wave == 0 && lane < LPR) {
#pragma unroll
        for (int w = 1; w < VEC_WAVES; w++) {
            RowPartial o;
            o.m = sh[w][lane][0];
            o.l = sh[w][lane][1];
#pragma unroll
            for (int e = 0; e < 8; e++) o.acc[e] = sh[w][lane][2 + e];
            row_partial_merge(st, o);
        }
        if (a.counters) row_store<LPR, true>(a, st, row, split, lane);
        else            row_store<LPR>(a, st, row, split, lane);
    }
    // the last of the row's n_splits workgroups merges them: no launch for the merge
    if (a.n_splits > 1 && a.counters) {
        __shared__ int last;
        if (fattn_last_of_set(a, row, a.n_splits, &last, false) && tid < a.D / 4) fattn_merge_row<true>(a, row, tid);
    }
}

template <int TYPE, int LPR>
__global__ void __launch_bounds__(VEC_THREADS) fattn_vec_kernel(const FattnArgs a) {
    // blockIdx.x = row * n_splits + split, row = (b*Nq + iq1)*Hq + h  (the dst row order)
    const int split = blockIdx.x % a.n_splits;
    const int row   = blockIdx.x / a.n_splits;
    const int h     = row % a.Hq;
    const int iq1   = (row / a.Hq) % a.Nq;
    const int b     = row / (a.Hq * a.Nq);
    const int hk    = h / a.gqa;
    const int bk    = b / a.bq;
    auto mask_of = [&]() __attribute__((always_inline)) {
        RowMaskTensor mask;
        mask.row   = a.mask ? (const uint16_t *)(a.mask + iq1 * a.nbm1 + (h % a.Hm) * a.nbm2 + (b % a.Bm) * a.nbm3) : nullptr;
        mask.slope = fattn_slope(a, h);
        return mask;
    };
    vec_body<TYPE, LPR, 0>(a, split, row, a.q + iq1 * a.nbq1 + h * a.nbq2 + b * a.nbq3, a.k + hk * a.nbk2 + bk * a.nbk3,
                           a.v + hk * a.nbv2 + bk * a.nbv3, mask_of, RowNothing());
}

// A decoder's step over F32 rows, or f16 rows of heads that the decode kernel does not take: one row a (head, sequence) or one
// sequence, no mask, no soft cap, every query head with keys of its own, K and V alike in their strides.  A call is a chain of latencies (arguments,
// the place in the grid, first requests, merges), and these are in it what they need to be: the numbers behind the requests are in
// registers when a wave starts (see ArgTail), a grid by range, head and row takes no division, and a lane asks for its part of a
// row in two pieces, all of a step's K and V before it looks at any.  The general form waits for q ahead of K, for K ahead of V (the
// compiler moves V's loads behind the branch that needs them), and at element-wise rows for each load of a branch.  us a call inside a
// graph, that form and this: 8 heads of 36 against 375 F32 rows 8.2 -> 5.4 (f16 10.7 -> 5.4), of 52 9.1 -> 5.4; 20 heads of 64 against 1500
// 10.2 -> 7.9, 16 of 128 against 700 10.3 -> 7.2; 5 rows x 20 heads of 52 against 1500 f16 rows 25.1 -> 8.3, 24 rows x 20 of 36 against 1500
// F32 rows 55.9 -> 14.7.
struct VecShort {
    const char * k;
    const char * v;
    const char * q;
    uint32_t     nbk1, nbk2, nbkz;    // and V's; z: of the sequence (0: one for all)
    uint32_t     nbq2, nbqz;          // z: of the row or of the sequence, whichever there are several of
    uint32_t     keys;                // Nkv | D / 4 << 25
    uint32_t     keys_per_split;
    float        scale;
    float *      dst;
    float *      part_acc;            // the (max, sum) pairs lie right behind it
    unsigned *   counters;
    uint32_t     Hq, n_splits, rows;
    uint32_t     unused;
    template <typename F> __host__ __device__ void pointers(F f) { f(k, v, q, dst, part_acc, counters); }
};
static_assert(sizeof(VecShort) == 96 && offsetof(VecShort, dst) == 56, "see above");

// 0: the call needs the wide form, else its PIECES
int vec_shorten(const FattnArgs & a, int ktype, VecShort & p) {
    const int64_t nb[9] = {a.nbk1, a.nbk2, a.nbk3, a.nbv1, a.nbv2, a.nbv3, a.nbq1, a.nbq2, a.nbq3};
    for (int64_t x : nb)
        if ((uint64_t)x > 0xFFFFFFFFull) return 0;
    if (a.mask || a.softcap != 0.0f || a.gqa != 1 || a.Dv != a.D || (a.Nq != 1 && a.B != 1) || !(a.Bk == 1 || a.Bk == a.B)) return 0;
    if (a.nbk1 != a.nbv1 || a.nbk2 != a.nbv2 || (a.Bk > 1 && a.nbk3 != a.nbv3)) return 0;
    const int64_t rows = (int64_t)a.Nq * a.Hq * a.B;
    if (a.Hq > 0xFFFF || a.Nq > 0xFFFF || a.B > 0xFFFF || rows > 0x7fffffff || a.Nkv < 1 || a.Nkv >= 1 << 25 || (int64_t)(a.n_splits - 1) * a.keys_per_split >= a.Nkv) return 0;      // (no range is empty)
    if (a.n_splits > 1 && a.part_ml != a.part_acc + rows * a.n_splits * a.D) return 0;
    if ((int64_t)a.Nkv * a.nbk1 + 1024 > 0xFFFFFFE0LL) return 0;             // a head's rows as one buffer
    // whole pieces of 4 elements, and q's of 16 bytes
    const int pieces = a.aligned16 && a.D % 8 == 0 ? 2 : 1;
    const uintptr_t unit = ktype == MI355X_TYPE_F32 ? 16 : 8;
    if (!a.q_aligned16 || ((uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.nbk1 | (uintptr_t)a.nbk2 | (a.Bk > 1 ? (uintptr_t)a.nbk3 : 0)) % unit) return 0;
    p.k = a.k; p.v = a.v; p.q = a.q; p.dst = a.dst;
    p.nbk1 = (uint32_t)a.nbk1; p.nbk2 = (uint32_t)a.nbk2; p.nbkz = a.Bk > 1 ? (uint32_t)a.nbk3 : 0;
    p.nbq2 = (uint32_t)a.nbq2; p.nbqz = (uint32_t)(a.B > 1 ? a.nbq3 : a.nbq1);
    p.keys = (uint32_t)a.Nkv | (uint32_t)a.D / 4 << 25; p.keys_per_split = (uint32_t)a.keys_per_split; p.Hq = (uint32_t)a.Hq;
    p.part_acc = a.n_splits > 1 ? a.part_acc : nullptr;
    p.counters = a.n_splits > 1 ? a.counters : nullptr;
    p.scale = a.scale;
    p.n_splits = (uint32_t)a.n_splits; p.rows = (uint32_t)rows; p.unused = 0;
    return pieces;
}

template <int TYPE, int LPR, int PIECES>
__global__ void __launch_bounds__(VEC_THREADS) __attribute__((amdgpu_waves_per_eu(4))) fattn_vec_short_kernel(FATTN_HEAD_PARAMS, const ArgTail<VecShort> tail) {
    const VecShort p = fattn_join<VecShort>(FATTN_HEAD_ARGS, tail);
    FattnArgs a = {};
    a.D = a.Dv = (int)(p.keys >> 25) * 4;
    a.Nq = (int)p.rows; a.Hq = a.B = 1;          // (the merge asks for the number of rows alone)
    a.Nkv = (int)(p.keys & 0x1FFFFFFu);
    a.n_splits = (int)p.n_splits;
    a.keys_per_split = (int)p.keys_per_split;
    a.nbk1 = a.nbv1 = p.nbk1;
    a.scale = p.scale;
    a.dst = p.dst;
    a.part_acc = p.part_acc;
    a.part_ml  = p.part_acc + (int64_t)p.rows * p.n_splits * a.D;
    a.counters = p.counters;
    const uint32_t h = blockIdx.y, z = blockIdx.z;
    const int64_t  kv = (int64_t)((uint64_t)h * p.nbk2 + (uint64_t)z * p.nbkz);
    auto no_mask = [&]() __attribute__((always_inline)) { return RowMaskTensor{nullptr, 0.0f}; };
    vec_body<TYPE, LPR, PIECES>(a, blockIdx.x, (int)(z * p.Hq + h), p.q + ((uint64_t)h * p.nbq2 + (uint64_t)z * p.nbqz), p.k + kv, p.v + kv, no_mask, [&]() __attribute__((always_inline)) {
                                    // the rest of the arguments arrives beside the first rows, not behind them
                                    asm volatile("" ::"s"(p.dst), "s"(p.part_acc), "s"(p.counters), "s"(p.Hq), "s"(p.n_splits), "s"(p.rows) : "memory");
                                });
}

// One row per D/4 lanes (a float4 of d each), 64 / (D/4) rows per wave.
__global__ void __launch_bounds__(256) fattn_merge_kernel(const FattnArgs a, int rows) {
    const int lpr  = a.D / 4;                       // lanes per row
    const int rpw  = 64 / lpr;                      // rows per wave
    const int lane = threadIdx.x & 63;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int row  = wave * rpw + lane / lpr;
    if (lane >= rpw * lpr || row >= rows) return;
    fattn_merge_row<false>(a, row, lane % lpr);
}

template <int TYPE>
int launch_typed(const FattnArgs & a, hipStream_t stream) {
    const int64_t rows = (int64_t)a.Nq * a.Hq * a.B;
    if (rows * a.n_splits > 0x7fffffff) return (int)hipErrorInvalidValue;      // one workgroup per (row, split)
    const dim3 grid((unsigned)(rows * a.n_splits));
    const dim3 block(VEC_THREADS);
    const int  lanes = (a.D + 7) / 8;
    if constexpr (TYPE == MI355X_TYPE_F32 || TYPE == MI355X_TYPE_F16) {
        VecShort  p;
        const int pieces = vec_shorten(a, TYPE, p);
        if (pieces) {
            const dim3 by((unsigned)a.n_splits, (unsigned)a.Hq, (unsigned)(a.Nq * a.B));
            auto go = [&](auto lpr) {
                constexpr int L = decltype(lpr)::value;
                if constexpr (TYPE == MI355X_TYPE_F16) {         // (F32 rows come in the same two loads either way)
                    if (pieces == 2) {
                        fattn_launch_head(fattn_vec_short_kernel<TYPE, L, 2>, by, block, 0, stream, p);
                        return;
                    }
                }
                fattn_launch_head(fattn_vec_short_kernel<TYPE, L, 1>, by, block, 0, stream, p);
            };
            if (lanes <= 4)       go(std::integral_constant<int, 4>{});
            else if (lanes <= 8)  go(std::integral_constant<int, 8>{});
            else if (lanes <= 16) go(std::integral_constant<int, 16>{});
            else                  go(std::integral_constant<int, 32>{});
            return (int)hipGetLastError();
        }
    }
    if (lanes <= 4)       fattn_launch((fattn_vec_kernel<TYPE, 4>),  grid, block, 0, stream, a);
    else if (lanes <= 8)  fattn_launch((fattn_vec_kernel<TYPE, 8>),  grid, block, 0, stream, a);
    else if (lanes <= 16) fattn_launch((fattn_vec_kernel<TYPE, 16>), grid, block, 0, stream, a);
    else                  fattn_launch((fattn_vec_kernel<TYPE, 32>), grid, block, 0, stream, a);
    return (int)hipGetLastError();
}

}  // namespace

int fattn_vec_launch(const FattnArgs & a, int ktype, hipStream_t stream) {
    switch (ktype) {
        case MI355X_TYPE_F16:  return launch_typed<MI355X_TYPE_F16>(a, stream);
        case MI355X_TYPE_F32:  return launch_typed<MI355X_TYPE_F32>(a, stream);
        case MI355X_TYPE_Q8_0: return launch_typed<MI355X_TYPE_Q8_0>(a, stream);
        case MI355X_TYPE_Q4_0: return launch_typed<MI355X_TYPE_Q4_0>(a, stream);
        case MI355X_TYPE_Q4_1: return launch_typed<MI355X_TYPE_Q4_1>(a, stream);
        case MI355X_TYPE_Q5_0: return launch_typed<MI355X_TYPE_Q5_0>(a, stream);
        case MI355X_TYPE_Q5_1: return launch_typed<MI355X_TYPE_Q5_1>(a, stream);
        default:               return (int)hipErrorInvalidValue;
    }
}

int fattn_vec_form(const FattnArgs & a, int ktype) {
    VecShort p;
    return (ktype == MI355X_TYPE_F32 || ktype == MI355X_TYPE_F16) && vec_shorten(a, ktype, p) ? MI355X_FATTN_FORM_SHORT : MI355X_FATTN_FORM_GENERAL;
}

int fattn_merge_launch(const FattnArgs & a, hipStream_t stream) {
    const int rows = a.Nq * a.Hq * a.B;
    const int rows_per_block = 4 * (64 / (a.D / 4));          // D is a multiple of 8, at most 256
    const dim3 grid((unsigned)((rows + rows_per_block - 1) / rows_per_block));
    fattn_launch(fattn_merge_kernel, grid, dim3(256), 0, stream, a, rows);
    return (int)hipGetLastError();
}
