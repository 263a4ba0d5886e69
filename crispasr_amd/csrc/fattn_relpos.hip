// FastConformer's relative-position attention in one kernel (the flash branch of core_conformer::build_block,
// src/core/fastconformer.h:876-934):
//
//   dst[:, h, i, b] = softmax_j( scale * <q_u[i], k[j]> + mask[j, i] ) . v[j]
//   mask[j, i]      = f16( scale * <q_v[i], r[Nq-1+j-i]> + add[j, i] )         (the graph's rel_shift view, scale, add, cast)
//
// The reference materialises `mask` as an F16 [T, T, H] tensor per sequence and hands it to ggml_flash_attn_ext; here
// the position term is produced tile by tile inside the attention loop and never leaves the CU.
//
// A workgroup of 2 to 4 waves owns consecutive queries of one (head, batch), 32 per wave (the N columns of
// v_mfma_f32_32x32x16_f16 accumulators), and walks the keys 32 at a time.  Per tile of keys and wave:
//   S^T  = K tile . Q_u^T                       8 (D = 128) MFMAs, A = K rows from LDS, B = Q_u in registers
//   BD   = R block . Q_v^T                      8 MFMAs, A = 32 rows of the table from LDS, B = Q_v in registers.
//          Block n x the wave's 32 queries is one accumulator whose element (row, il) belongs to key
//          j = 32 n + row + il - 31: tile t is the lower-right triangle (row + il >= 31) of block t and the upper-left
//          one of block t + 1, and for one accumulator slot exactly one of the two owns the slot's place in the tile -
//          so the previous block stays in registers, one new block is computed per step and a select per slot gives
//          the tile, each product computed once.
//   un-skew: the selected values sit at key (row + il + 1) mod 32 of their query; they go through a wave-private
//          32 x 32 f32 square in LDS (pitch 36: writes and the 16-byte row reads are both conflict-free) and come back
//          in the layout of S^T.
//   mask = f16(scale * BD + add), s = S + mask in log2 units, online softmax against a reference that is raised
//          only when the 16 probabilities of a lane sum to more than FR_SUM_LIMIT, P -> f16
//   O^T += V^T . P^T                            8 MFMAs, A = V tile through ds_read_b64_tr_b16, B = P from registers
// The waves need the same table rows one step apart, so the table is staged once per workgroup in a ring of 32-row blocks,
// one more than there are waves.  K and V tiles and table blocks move global -> LDS without passing registers (16 bytes a lane, the
// chunks of a row XOR-swizzled so that the operand reads are conflict-free; in the loop by buffer loads, a tensor's buffer
// ending with its last row).  The step of tile t requests K tile t + 2, table block t + 3 and V tile t + 1, which the next step reads, into
// the halves and the slot that the step before it has left - K and V have two halves each - and one barrier at its end waits for
// them.  K, V and the table are f16 with 16-byte aligned rows (the caller rounds F32 ones first, as the reference's own graph does
// for the mask product's operands).
//
// The vector work of a tile stands beside the matrix instructions of another: a step turns tile t's scores into probabilities beside
// the two Q products of tile t + 1, and un-skews those beside P.V.  Q_u, Q_v and the result pass through the wave's square, so that
// the memory sees them along the rows.
//
// What bounds it: the blocks of a step are requested one step ahead, and its waves walk the keys in phase, so that each waits for
// its first reader's trip to memory (8 x 8 heads of 128 x 750, two workgroups of 3 waves a CU: 70 us, 61 without the loop's
// requests, 57 without its mask either); 40 us are ahead of the second step and behind the last, 13 of them Q_u's and Q_v's.
// Against all of a step in one chain, operands of Q fetched as they lie and requests of six instructions, us a call: 8 heads x
// 128, 300 tokens 22.9 -> 19.6, 120 x 8 16.9 -> 14.7, 200 x 4 22.5 -> 20.6, 1000 x 2 55.2 -> 48.7, 750 x 8 (F32 K, V and table) 88.1 -> 85.6;
// 8 x 64, 750 x 8 46.5 -> 45.9.  Registers are short in the 128-wide forms with a mask: one spilled operand is a load whose wait
// takes the requests in with it (+5 us at 1000 x 2), which is why sums of addresses are kept from moving out of the loop.
#include "fattn_row.h"

#include <stdlib.h>
#include <type_traits>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float    float2v __attribute__((ext_vector_type(2)));
typedef float    float16v __attribute__((ext_vector_type(16)));
typedef float    float4v __attribute__((ext_vector_type(4)));
typedef short    short4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float    float4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 half4_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int   FR_SQP   = 36;                      // pitch of the un-skew square in floats
constexpr float FR_LOG2E = 1.4426950408889634f;
constexpr float FR_SUM_LIMIT = 4096.0f;               // a tile's 16 probabilities of a lane sum to at most this before the reference is raised

template <int D> constexpr int fr_kp() { return 2 * D; }          // bytes per K / table row in LDS (chunks swizzled, no padding)
template <int D> __device__ __forceinline__ int fr_swz(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
template <int D> __device__ __forceinline__ int fr_swz_v(int r) { return D == 64 ? r & 7 : (r & 3) << 2; }
// what stands before it stays there, what stands behind it too
#define FR_FENCE() __builtin_amdgcn_sched_barrier(0)
constexpr int FR_RD = 3, FR_VD = 2;                   // operands of the two Q products and of P.V that are read ahead (four: scratch)
// two K tiles, two V tiles, NW + 1 table blocks (NW in use, one being written), one un-skew square per wave
template <int D, int NW> constexpr int fr_lds_bytes() { return (4 + NW + 1) * 32 * fr_kp<D>() + NW * 32 * FR_SQP * 4; }

template <int D, int NW, bool ADD, bool ADD_F16>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) fattn_relpos_kernel(const FattnRelposArgs a) {
    constexpr int FR_SLOTS = NW + 1;
    constexpr int KS  = D / 16;                     // reduction steps of the two Q products
    constexpr int DBO = D / 32;                     // 32-wide blocks of the output's d
    constexpr int CH  = D / 8;                      // 16-byte chunks per row
    constexpr int KP  = fr_kp<D>();

    extern __shared__ __attribute__((aligned(256))) char fr_lds[];
    char * const kt   = fr_lds;                     // tile t: half t % 2
    char * const vt   = kt + 2 * 32 * KP;
    char * const ring = vt + 2 * 32 * KP;
    const int tid  = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int il   = lane & 31;
    const int hh   = lane >> 5;
    float * const sq = (float *)(ring + FR_SLOTS * 32 * KP) + wave * 32 * FR_SQP;

    // Workgroups go to the 8 XCDs round-robin, each with its own L2: the query blocks of one (head, batch) are given to
    // one XCD, so that K, V and the table rows they share come from that L2.  The head index runs faster than the batch:
    // an XCD holds all heads of few sequences, which share the sequence's additive mask (2 MB at T = 750 in F32; with the
    // batch running faster every XCD fetched every sequence's mask and the call took 5% longer).
    const int     n_qb = (a.Nq + 32 * NW - 1) / (32 * NW);
    const int64_t G    = (int64_t)n_qb * a.H * a.B;
    const int64_t per  = (G + 7) / 8;
    const int64_t L    = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || L >= G) return;
    const int qb = (int)(L % n_qb);
    const int h  = (int)((L / n_qb) % a.H);
    const int b  = (int)(L / ((int64_t)n_qb * a.H));
    const int hk = h / a.gqa, bk = b / a.bq;

    const int q0  = qb * 32 * NW;
    const int i0w = q0 + wave * 32;
    const int iq  = min(i0w + il, a.Nq - 1);        // rows past Nq repeat the last one and are not stored
    const int NT  = (a.Nkv + 31) / 32;
    const int NR  = a.Nq + a.Nkv - 1;
    const int p_base0 = a.Nq - 1 - q0 - 31;         // table row of (block 0, row 0) in wave 0's numbering; wave w's block n is block n - w

    const char * kbase = a.k + (int64_t)hk * a.nbk2 + (int64_t)bk * a.nbk3;
    const char * vbase = a.v + (int64_t)hk * a.nbv2 + (int64_t)bk * a.nbv3;
    const char * rbase = a.r + (int64_t)(h % a.Hr) * a.nbr2 + (int64_t)(b % a.Br) * a.nbr3;

    // ---- staging ------------------------------------------------------------------------------------------------
    // K tiles and table blocks: each wave moves its quarter, 64 x 16 bytes per instruction; LDS slot
    // L = (wave * NDM + j) * 64 + lane holds chunk (L % CH) ^ swizzle of row L / CH.  Rows that stick out (the last key
    // tile, the ends of the table) repeat the nearest valid row: they belong to excluded keys or to no key at all.
    constexpr int TI  = 32 * CH * 16 / 1024;                  // 64-lane instructions per tile
    constexpr int NDM = (TI + NW - 1) / NW;                   // ... per wave: instruction j of wave w is number j * NW + w
    // Instruction number ins moves rows ins * RPI .. + RPI - 1: the lane's row and chunk in it are the same for every ins but
    // for one or two bits of the K layout's swizzle, so that an instruction's addresses cost two operations.
    constexpr int RPI = 64 / CH;
    const int      lr = lane / CH, lc = lane % CH;
    const uint32_t ck = (uint32_t)((lc ^ fr_swz<D>(lr)) * 16), cv = (uint32_t)((lc ^ fr_swz_v<D>(lr)) * 16);
    static_assert(RPI == 4 || RPI == 8, "the swizzles of rows r and r + RPI * ins differ by 4 * (ins % (16 / RPI)) (K) or not at all (V)");
    // Rows row0 .. row0 + 31 of a tensor, in one of two layouts, before the loop.  (NW = 3: the last wave repeats an instruction of
    // the one before.)
    auto dma_rows = [&](char * dst, const char * base, int64_t nb1, int row0, int last_row, bool is_v) __attribute__((always_inline)) {
        const uint32_t to    = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)dst;
        const uint32_t nb    = (uint32_t)nb1;                         // (row offsets inside a tile are 32-bit)
        const int      first = min(max(row0, 0), last_row);
        const uint64_t at    = (uint64_t)(base + (int64_t)first * nb1);
#pragma unroll
        for (int j = 0; j < NDM; j++) {
            const uint32_t ins = min((uint32_t)(j * NW + wave), (uint32_t)TI - 1);             // uniform
            const uint32_t rr  = (uint32_t)(min(max(row0 + (int)ins * RPI + lr, 0), last_row) - first);
            load_to_lds16<true>(at, rr * nb + (is_v ? cv : ck ^ ((ins & (16 / RPI - 1)) * 64)), to + ins * 1024);
        }
    };
    auto dma_k = [&](int t) __attribute__((always_inline)) { dma_rows(kt + (t & 1) * 32 * KP, kbase, a.nbk1, 32 * t, a.Nkv - 1, false); };
    auto dma_v = [&](int t) __attribute__((always_inline)) { dma_rows(vt + (t & 1) * 32 * KP, vbase, a.nbv1, 32 * t, a.Nkv - 1, true); };
    auto slot_of = [&](int beta) { return ring + ((beta + NW - 1) % FR_SLOTS) * 32 * KP; };   // beta >= 1 - NW
    auto dma_r = [&](int beta, char * to) __attribute__((always_inline)) { dma_rows(to, rbase, a.nbr1, p_base0 + 32 * beta, NR - 1, false); };

    // ---- prologue: table blocks 1 - NW .. 2, the first K tiles and V tile, Q_u and Q_v as B operands -----------------
    // (block 1 - NW, which only the last wave reads and only here, lies in V's second half: its slot has block 2 already; calls of one
    //  tile need neither that block nor the second K tile)
    char * const first_block = vt + 32 * KP;
    dma_r(1 - NW, first_block);
#pragma unroll 1
    for (int beta = 2 - NW; beta <= (NT > 1 ? 2 : 1); beta++) dma_r(beta, slot_of(beta));
    dma_k(0);
    dma_v(0);
    if (NT > 1) dma_k(1);
    // Q_u and Q_v come along the rows, 4 of 64 values an instruction, and turn into B operands in the wave's square, as f16: fetched as
    // the operands lie an instruction takes 32 bytes of each of 32 rows.  (Not 128-wide calls of one tile, whose results do not
    // take the square either: with one instruction's rows the way through LDS is what shows. 8 heads x 8 tokens 8.15 -> 7.55 us, x 17 8.45 -> 7.85,
    // x 32 8.45 -> 8.15, under an F16 mask 17 9.15 -> 8.65; under an F32 mask there are no registers for a second way.)
    constexpr bool ONE_TILE = D == 128 && (!ADD || ADD_F16);
    half8 qu[KS], qv[KS];
    if (ONE_TILE && NT == 1) {
        const float * pu = (const float *)(a.qu + (int64_t)iq * a.nbu1 + (int64_t)h * a.nbu2 + (int64_t)b * a.nbu3) + hh * 8;
        const float * pv = (const float *)(a.qv + (int64_t)iq * a.nbw1 + (int64_t)h * a.nbw2 + (int64_t)b * a.nbw3) + hh * 8;
        const float   qs = a.scale * FR_LOG2E;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int p4 = 0; p4 < 2; p4++) {
                const float4v u = *(const float4v *)(pu + ks * 16 + p4 * 4), w = *(const float4v *)(pv + ks * 16 + p4 * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    qu[ks][4 * p4 + e] = (_Float16)(u[e] * qs);
                    qv[ks][4 * p4 + e] = (_Float16)w[e];
                }
            }
    } else {
        constexpr int QP = D / 64;                                    // pieces of 64 values a row
        const int     qr = lane >> 4, qc = lane & 15;
        float4v       raw[2 * QP][8];
#pragma unroll
        for (int i = 0; i < 2 * QP; i++) {
            const bool    u  = i < QP;
            const char  * at = (u ? a.qu + (int64_t)h * a.nbu2 + (int64_t)b * a.nbu3 : a.qv + (int64_t)h * a.nbw2 + (int64_t)b * a.nbw3) + i % QP * 256 + qc * 16;
#pragma unroll
            for (int j = 0; j < 8; j++) raw[i][j] = *(const float4v *)(at + (int64_t)min(i0w + 4 * j + qr, a.Nq - 1) * (u ? a.nbu1 : a.nbw1));
        }
        const float qs = a.scale * FR_LOG2E;
#pragma unroll
        for (int i = 0; i < 2 * QP; i++) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                half4 x;
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = (_Float16)(i < QP ? raw[i][j][e] * qs : raw[i][j][e]);
                *(half4 *)((char *)sq + (4 * j + qr) * (FR_SQP * 4) + qc * 8) = x;
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int e = 0; e < 4; e++) (i < QP ? qu : qv)[i % QP * 4 + e] = *(const half8 *)((const char *)sq + il * (FR_SQP * 4) + e * 32 + hh * 16);
            asm volatile("" ::: "memory");
        }
    }
    constexpr int AES = ADD_F16 ? 2 : 4;
    uint32_t add_off = 0;                           // the query's row of the additive mask, from that of the wave's first query
    // (The head's and the sequence's offsets in scalar registers: the divisions leave theirs in vector ones, and the 128-wide
    //  forms held them through the loop in scratch, for the rows that are done again.)
    const char * add_head = nullptr, * add_wave = nullptr;
    if (ADD) {
        add_head = a.add + (int64_t)__builtin_amdgcn_readfirstlane(h % a.Ha) * a.nba2 + (int64_t)__builtin_amdgcn_readfirstlane(b % a.Ba) * a.nba3;
        add_wave = add_head + (int64_t)min(i0w, a.Nq - 1) * a.nba1;
        add_off  = (uint32_t)(iq - min(i0w, a.Nq - 1)) * (uint32_t)a.nba1;
    }
    // the additive mask's values of a tile: requested when the tile before is done with its own, waited for with that
    // tile's blocks
    typedef typename std::conditional<ADD_F16, half4_a2, float4_a4>::type araw_t;
    araw_t araw[ADD ? 4 : 1];
    auto load_add = [&](int t) __attribute__((always_inline)) {
        const char * tile = add_wave + (int64_t)32 * AES * t;                                 // uniform
        uint32_t off = add_off;
        int      key = 4 * hh;
        asm volatile("" : "+v"(off), "+v"(key));              // (sums of them are not worth registers in the loop)
        if (__builtin_expect(32 * t + 32 <= a.Nkv, 1)) {
#pragma unroll
            for (int g = 0; g < 4; g++) araw[ADD ? g : 0] = *(const araw_t *)(tile + (off + key * AES) + 8 * g * AES);
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const uint32_t at = off + (uint32_t)min(8 * g + key + c, a.Nkv - 1 - 32 * t) * AES;
                    if constexpr (ADD_F16) araw[ADD ? g : 0][c] = *(const _Float16 *)(tile + at);
                    else                   araw[ADD ? g : 0][c] = *(const float *)(tile + at);
                }
        }
    };
    // (the first tile's with the first blocks: behind the barrier they were a round trip of their own, 0.2 us of a call of two
    //  tiles - 50 tokens x 4 heads of 64 7.6 -> 7.4 us)
    if (ADD) load_add(0);
    // Keys beyond the length of a padded sequence carry -inf in the additive mask for every query: tiles that are masked
    // out entirely at the END of the key range add nothing and are not walked at all.  Each wave looks at its queries'
    // last tile while the first blocks are on their way (that is all an unpadded sequence costs) and, if that one is
    // masked, scans backwards four tiles per round trip; the workgroup takes the largest count.
    int NTL = NT;
    if (ADD) {
        const int tr = lane >> 3, tc = (lane & 7) * 4;                // (along the rows: 8 of them an instruction)
        auto tile_max = [&](int tt) __attribute__((always_inline)) {
            float v = -INFINITY;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const char * row = add_head + (int64_t)min(i0w + 8 * g + tr, a.Nq - 1) * a.nba1;
                const int key0 = 32 * tt + tc;
                if (32 * tt + 32 <= a.Nkv) {
                    if (ADD_F16) {
                        const half4_a2 x = *(const half4_a2 *)(row + (int64_t)key0 * 2);
                        v = fmaxf(fmaxf(v, fmaxf((float)x[0], (float)x[1])), fmaxf((float)x[2], (float)x[3]));
                    } else {
                        const float4_a4 x = *(const float4_a4 *)(row + (int64_t)key0 * 4);
                        v = fmaxf(fmaxf(v, fmaxf(x[0], x[1])), fmaxf(x[2], x[3]));
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const int key = min(key0 + c, a.Nkv - 1);
                        v = fmaxf(v, ADD_F16 ? (float)*(const _Float16 *)(row + (int64_t)key * 2) : *(const float *)(row + (int64_t)key * 4));
                    }
                }
            }
            return v;
        };
        auto any_live = [&](float v) { return __builtin_amdgcn_ballot_w64(v > -INFINITY || v != v) != 0; };
        int live = NT;
        if (NT > 1 && !any_live(tile_max(NT - 1))) {
            live = NT - 1;
            while (live > 0) {
                const int t0 = max(live - 4, 0);
                float mx[4];
#pragma unroll
                for (int u = 0; u < 4; u++) mx[u] = tile_max(min(t0 + u, live - 1));
                unsigned bits = 0;
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (any_live(mx[u])) bits |= 1u << u;
                if (bits) {
                    live = min(t0 + (32 - __builtin_clz(bits)), live);
                    break;
                }
                live = t0;
            }
        }
        // (the four floats behind each row of a square are padding that nothing else writes)
        if (lane == 0) ((int *)(ring + FR_SLOTS * 32 * KP))[32 + wave] = live;
    }
    // every wave's share of what it requested is in LDS, and every wave is done with what it read there
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    meet();
    if (ADD) {
        NTL = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) NTL = max(NTL, ((const int *)(ring + FR_SLOTS * 32 * KP))[32 + w]);
    }

    // operand reads of a K or table block: lane (il, hh) takes d = 16 ks + 8 hh .. +7 of row il.  (Tiles and blocks lie at
    // multiples of their size, so the address of operand ks is that of operand 0 with the bits of ks turned over.)
    const uint32_t op0 = (uint32_t)((il * CH + (hh ^ fr_swz<D>(il))) * 16);
    // transposing reads of the V tile: lane j16 of a group of 16 addresses key 4 hh + j16 / 4 (+ 8, + 16 ks) and four
    // values of d from 32 db + 16 (group % 2) + 4 (j16 % 4) on; the swizzle depends on key % 8 only
    uint32_t va0;
    {
        const int j16 = lane & 15, G16 = lane >> 4, kr0 = 4 * (G16 >> 1) + (j16 >> 2);
        const int c = 2 * (G16 & 1) + ((j16 & 3) >> 1);
        va0 = (uint32_t)((kr0 * CH + (c ^ fr_swz_v<D>(kr0))) * 16 + 8 * (j16 & 1));
    }
    typedef __attribute__((address_space(3))) const half8 lds_half8;
    typedef __attribute__((address_space(3))) short4v lds_short4;
    auto lds_at = [&](const char * p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)p; };

    auto read_block = [&](half8 (&to)[KS], const char * blk) __attribute__((always_inline)) {
        const uint32_t at = lds_at(blk) + op0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) to[ks] = *(lds_half8 *)(uintptr_t)(at ^ (ks * 32));
    };
    auto times_q = [&](const half8 (&block)[KS], const half8 (&q)[KS]) __attribute__((always_inline)) {
        float16v acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(block[ks], q[ks], acc, 0, 0, 0);
        return acc;
    };

    float16v oacc[DBO];
#pragma unroll
    for (int db = 0; db < DBO; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[db][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;

    // un-skew: slot r of a lane sits at row k_r + 4 hh of its block, i.e. at key (x + k_r) mod 32 with x = il + 4 hh + 1, and
    // belongs to the previous block exactly when that sum reaches 32
    const int x_lane = il + 4 * hh + 1;
    int sq_new = il * FR_SQP + x_lane;
    auto unskew = [&](int r, const float16v & older, const float16v & newer) __attribute__((always_inline)) {
        const int  k_r  = 8 * (r >> 2) + (r & 3);
        const bool prev = x_lane + k_r >= 32;
        sq[(prev ? sq_new - 32 : sq_new) + k_r] = prev ? older[r] : newer[r];
    };
    float4v bd[4];                                     // a tile's position scores, back in the layout of S^T
    auto read_square = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 4; g++) bd[g] = *(const float4v *)&sq[il * FR_SQP + 8 * g + 4 * hh];
    };

    // the first tile's products: the wave's blocks 0 (= block -wave in wave 0's numbering), whose lower-right triangle it takes, and 1
    float16v bd_prev, s;
    {
        half8 ops[KS];
        read_block(ops, wave == NW - 1 ? first_block : slot_of(-wave));
        const float16v bd0 = times_q(ops, qv);
        read_block(ops, slot_of(1 - wave));
        bd_prev = times_q(ops, qv);
        read_block(ops, kt);
        s = times_q(ops, qu);
#pragma unroll
        for (int r = 0; r < 16; r++) unskew(r, bd0, bd_prev);
        read_square();
    }

    // (the compiler's wait for them belongs here, behind that of `meet`: further down it would wait for the blocks on their way)
    auto have_add = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 4; g++) asm volatile("" : "+v"(araw[ADD ? g : 0]));
    };
    meet();                                            // what was read here may be written over
    if (ADD) have_add();

    // A step's requests, K tile t + 2, table block t + 3 and V tile t + 1: workgroups of 3 waves share them out by tensor, 8 or 4 to
    // each, others by rows, so that a wave's are as many as any other's.  A tensor's rows of one step are a buffer that ends
    // with the tensor's last row (rows behind it are zeros: excluded keys, or no key at all), its address moves on by 32 rows.
    constexpr bool BY_TENSOR = NW == 3;
    constexpr int  TPW = BY_TENSOR ? 1 : 3, IPT = BY_TENSOR ? TI : TI / NW;        // tensors of a wave, instructions of each
    uint64_t rq_base[TPW];
    uint32_t rq_nb[TPW], rq_row[TPW], rq_chunk[TPW];   // pitch; the lane's row and chunk in an instruction
    int      rq_left[TPW];                             // rows from the step's first one on
    const uint32_t rq_ins = BY_TENSOR ? 0 : (uint32_t)wave;
    constexpr uint32_t RQ_STRIDE = BY_TENSOR ? 1 : NW;
#pragma unroll
    for (int i = 0; i < TPW; i++) {
        const int      which = BY_TENSOR ? wave : i;
        const int      row0  = which == 0 ? 64 : which == 1 ? p_base0 + 96 : 32;
        const int64_t  nb1   = which == 0 ? a.nbk1 : which == 1 ? a.nbr1 : a.nbv1;
        rq_base[i]  = (uint64_t)((which == 0 ? kbase : which == 1 ? rbase : vbase) + (int64_t)row0 * nb1);
        rq_nb[i]    = (uint32_t)nb1;
        rq_left[i]  = (which == 1 ? NR : a.Nkv) - row0;
        rq_row[i]   = (uint32_t)lr * rq_nb[i];
        rq_chunk[i] = which == 2 ? cv : ck;
    }
    constexpr int NRQ = TPW * IPT;
    __amdgpu_buffer_rsrc_t rq_buf[TPW];
    uint32_t rq_to[TPW];
    const uint32_t lds_k = lds_at(kt), lds_v = lds_at(vt), lds_ring = lds_at(ring);
    uint32_t ring_next = (uint32_t)(3 + NW - 1) % FR_SLOTS;                   // slot of block t + 3
    auto requests_of = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TPW; i++) {
            const int      which = BY_TENSOR ? wave : i;
            const int      rows  = min(rq_left[i], 32);
            rq_buf[i]   = fattn_buffer((const void *)rq_base[i], rows > 0 ? (uint32_t)(rows - 1) * rq_nb[i] + 2 * D : 0);
            rq_base[i] += (uint64_t)rq_nb[i] * 32;
            rq_left[i] -= 32;
            asm volatile("" : "+v"(rq_row[i]), "+v"(rq_chunk[i]));           // (their sums are not worth registers in the loop)
            rq_to[i]    = which == 0 ? lds_k + (t & 1) * 32 * KP : which == 1 ? lds_ring + ring_next * 32 * KP : lds_v + ((t + 1) & 1) * 32 * KP;
        }
        ring_next = ring_next + 1 == FR_SLOTS ? 0 : ring_next + 1;
    };
    auto request = [&](int n) __attribute__((always_inline)) {
        const int      i    = n / IPT, j = n % IPT;
        const uint32_t ins  = rq_ins + j * RQ_STRIDE;
        const uint32_t turn = (BY_TENSOR ? wave : i) == 2 ? 0 : (ins & (16 / RPI - 1)) * 64;
        const uint32_t off  = (rq_chunk[i] ^ turn) + rq_row[i] + ins * RPI * rq_nb[i];
        buffer_to_lds16(rq_buf[i], off, rq_to[i], ins * 1024);
    };

    // A step turns the scores of tile t, which the step before has left in registers, into probabilities beside the products of tile t + 1,
    // and un-skews those beside P.V: a matrix instruction is followed by its share of the vector work, its next operand and a request,
    // and none of them moves (FR_FENCE).  The last step stands by itself, without products and requests: as a turn of the loop like the
    // others it took 0.6 to 0.9 us more, 8% of a call of 50 tokens (8 x 64 8.5 -> 7.7 us, 8 x 128 10.4 -> 9.6; 1000 tokens x 4 heads of 64 x 8 47.1 -> 46.0).
    uint32_t ring_at = (uint32_t)(2 - wave + NW - 1) % FR_SLOTS;              // slot of the wave's block t + 2
    auto step = [&](int t, auto more) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        if (MORE) requests_of(t);
        constexpr int OPS = 2 * KS, RD = FR_RD, PER = 16 / OPS;               // products; operands read ahead; pairs of scores to each
        const uint32_t r_at = lds_ring + ring_at * 32 * KP + op0, k_at = lds_k + ((t + 1) & 1) * 32 * KP + op0;
        ring_at = ring_at + 1 == FR_SLOTS ? 0 : ring_at + 1;
        auto operand = [&](int i) __attribute__((always_inline)) { return *(lds_half8 *)(uintptr_t)((i < KS ? r_at : k_at) ^ (i % KS * 32)); };
        half8 ops[RD];
#pragma unroll
        for (int i = 0; i < (MORE ? RD : 0); i++) ops[i] = operand(i);
        FR_FENCE();
        float16v acc = {};
        auto product = [&](int i) __attribute__((always_inline)) {
            if (!MORE) return;
            if (i % KS == 0) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[r] = 0.0f;
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ops[i % RD], i < KS ? qv[i % KS] : qu[i % KS], acc, 0, 0, 0);
            if (i + RD < OPS) ops[i % RD] = operand(i + RD);
#pragma unroll
            for (int n = NRQ * i / OPS; n < NRQ * (i + 1) / OPS; n++) request(n);
        };
        // ---- mask = f16(scale * BD + add); scores in log2 units ------------------------------------------------------
        float s2[16];
        auto mask_pair = [&](int r) __attribute__((always_inline)) {
            float2v mk;
#pragma unroll
            for (int e = 0; e < 2; e++)                        // as the graph: scale, then add
                mk[e] = ADD ? mul_then_add(bd[r >> 2][(r & 3) + e], a.scale, (float)araw[ADD ? r >> 2 : 0][(r & 3) + e]) : bd[r >> 2][(r & 3) + e] * a.scale;
            uint32_t pk;                                       // rounded two at a time (the compiler converts one at a time)
            asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(pk) : "v"(mk[0]), "v"(mk[1]));
            const half2v mh = __builtin_bit_cast(half2v, pk);
#pragma unroll
            for (int e = 0; e < 2; e++) s2[r + e] = fmaf((float)mh[e], FR_LOG2E, s[r + e]);
        };
#pragma unroll
        for (int i = 0; i < KS; i++) {
            product(i);
#pragma unroll
            for (int n = 0; n < PER; n++) mask_pair(2 * (i * PER + n));
            FR_FENCE();
        }
        const float16v bd_new = acc;
        if (ADD && MORE) load_add(t + 1);
        if (__builtin_expect(32 * t + 32 > a.Nkv, 0)) {    // keys past the end of the last tile
            int key = 4 * hh;
            asm volatile("" : "+v"(key));
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (key + 8 * (r >> 2) + (r & 3) >= a.Nkv - 32 * t) s2[r] = -INFINITY;
        }

        // ---- online softmax ----------------------------------------------------------------------------------------------
        // P = 2^(s2 - m) in f16 against the row's reference m as it stands; the row sum is taken over the rounded values
        // the MFMA will use.  No maximum is computed on this path: a reference that has fallen too far behind shows up as
        // a large (or infinite, or NaN) tile sum, and only then - and on a row's first step - is the tile done again
        // with the reference raised to the tile's maximum.  Sums and accumulators are f32; a probability stays below
        // FR_SUM_LIMIT in f16.
        half8 p[2];
        float lsum = 0.0f;
        auto exp_pair = [&](int r, float ref) __attribute__((always_inline)) {
            const half2v ones = {(_Float16)1.0f, (_Float16)1.0f};
            half2v p2;
            p2[0] = (_Float16)__builtin_amdgcn_exp2f(s2[r] - ref);
            p2[1] = (_Float16)__builtin_amdgcn_exp2f(s2[r + 1] - ref);
            lsum = __builtin_amdgcn_fdot2(p2, ones, lsum, false);
            p[r >> 3][r & 7]       = p2[0];
            p[r >> 3][(r & 7) + 1] = p2[1];
        };
        {
            const float ref = m == -INFINITY ? 0.0f : m;
#pragma unroll
            for (int i = 0; i < KS; i++) {
                product(KS + i);
#pragma unroll
                for (int n = 0; n < PER; n++) exp_pair(2 * (i * PER + n), ref);
                FR_FENCE();
            }
        }
        s = acc;
        // ---- O^T += V^T . P^T -------------------------------------------------------------------------------------------
        constexpr int VOPS = 2 * DBO, VD = FR_VD;
        const uint32_t v_at = lds_v + (t & 1) * 32 * KP + va0;
        auto v_operand = [&](int i) __attribute__((always_inline)) {
            const uint32_t p0 = (v_at ^ (i / 2 * 64)) + 16 * (i % 2) * KP;
            const half4 lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(uintptr_t)p0));
            const half4 hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(uintptr_t)(p0 + 8 * KP)));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        half8 vops[VD];
#pragma unroll
        for (int i = 0; i < VD; i++) vops[i] = v_operand(i);
        if (__builtin_amdgcn_ballot_w64(!(lsum <= FR_SUM_LIMIT) || m == -INFINITY) != 0) {     // wave-uniform; rare after the first step
            float tmax = s2[0];
#pragma unroll
            for (int r = 1; r < 16; r++) tmax = fmaxf(tmax, s2[r]);
            tmax = max_of_halves(tmax);                        // both halves of a query must agree
            const float mn = tmax > m ? tmax : m;
            const float f  = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);     // m = -inf: nothing accumulated yet, f = 0
            l *= f;
#pragma unroll
            for (int db = 0; db < DBO; db++) oacc[db] *= f;
            m = mn;
            const float ref = m == -INFINITY ? 0.0f : m;
            lsum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                exp_pair(r, ref);
                FR_FENCE();                                    // (a pair at a time: there are no registers for more)
            }
        }
        l += lsum;
        asm volatile("" : "+v"(sq_new));                   // (nor are the slots' addresses)
        FR_FENCE();
#pragma unroll
        for (int i = 0; i < VOPS; i++) {
            oacc[i / 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vops[i % VD], p[i % 2], oacc[i / 2], 0, 0, 0);
            if (i + VD < VOPS) vops[i % VD] = v_operand(i + VD);
#pragma unroll
            for (int r = 16 * i / VOPS; r < 16 * (i + 1) / VOPS; r++) if (MORE) unskew(r, bd_prev, bd_new);
            FR_FENCE();
        }
        if constexpr (MORE) {
            bd_prev = bd_new;
            read_square();
            meet();
            if (ADD) have_add();
        }
    };
#pragma unroll 1
    for (int t = 0; t < NTL - 1; t++) step(t, std::true_type{});
    if (NTL > 0) step(NTL - 1, std::false_type{});

    // ---- normalise and store: lane (il, hh) holds d = 32 db + 8 g + 4 hh + c of its query -------------------------------
    l = sum_of_halves(l);
    // Excluded keys (add = -inf) were multiplied by probabilities of exactly zero, not skipped: the same for finite K/V, NaN
    // otherwise.  Queries whose result is not finite are computed again below, excluded keys unread, as the CPU op does it.
    uint64_t badbits = 0;
    if constexpr (ADD) {
        float chk = l * 0.0f;
#pragma unroll
        for (int db = 0; db < DBO; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) chk = fmaf(oacc[db][r], 0.0f, chk);
        badbits = __builtin_amdgcn_ballot_w64(chk != 0.0f);
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    auto value4 = [&](int db, int g) __attribute__((always_inline)) {
        float4v o;
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = oacc[db][4 * g + c] * inv;
        return o;
    };
    if (D == 64 || (ONE_TILE && NT == 1)) {
        // (as they lie: the way through the square costs these short calls 0.1 to 0.2 us, 33 tokens x 8 heads 7.65 and 7.45)
        if (i0w + il < a.Nq) {
            float * const out = a.dst + (((int64_t)b * a.Nq + (i0w + il)) * a.H + h) * D;
#pragma unroll
            for (int db = 0; db < DBO; db++)
#pragma unroll
                for (int g = 0; g < 4; g++) *(float4v *)(out + 32 * db + 8 * g + 4 * hh) = value4(db, g);
        }
    } else {   // through the square, 32 values of d at a time: 8 rows of 128 bytes a store instead of 32 bytes of 32 rows
        int         at   = lane;
        asm volatile("" : "+v"(at));                                  // (not worth registers in the loop)
        const int   orow = at >> 3, ocol = (at & 7) * 4;
        float * const out = a.dst + (((int64_t)b * a.Nq + i0w) * a.H + h) * D + ocol;
#pragma unroll
        for (int db = 0; db < DBO; db++) {
#pragma unroll
            for (int g = 0; g < 4; g++) *(float4v *)&sq[il * FR_SQP + 8 * g + 4 * hh] = value4(db, g);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4v o = *(const float4v *)&sq[(8 * j + orow) * FR_SQP + ocol];
                if (i0w + 8 * j + orow < a.Nq) *(float4v *)(out + (int64_t)(8 * j + orow) * a.H * D + 32 * db) = o;
            }
        }
    }
    if constexpr (ADD) {
        if (badbits != 0) {
            __threadfence();
            uint32_t bits = (uint32_t)badbits | (uint32_t)(badbits >> 32);      // lanes l and l + 32 hold the same query
            while (bits != 0) {
                const int qi = i0w + __builtin_ctz(bits);
                bits &= bits - 1;
                if (qi < a.Nq) attn_row_redo_relpos<D>(a, qi, h, b, add_head);
            }
        }
    }
}

template <int D, int NW>
int launch_d(const FattnRelposArgs & a, hipStream_t stream) {
    const int64_t G = (int64_t)((a.Nq + 32 * NW - 1) / (32 * NW)) * a.H * a.B;
    const int64_t grid = (G + 7) / 8 * 8;
    if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
    constexpr int lds = fr_lds_bytes<D, NW>();
#define FR_LAUNCH(ADD, F16)                                                                                                   \
    do {                                                                                                                      \
        static std::atomic<uint64_t> lds_allowed{0};                                                                          \
        const hipError_t e = fattn_allow_lds((const void *)fattn_relpos_kernel<D, NW, ADD, F16>, lds, lds_allowed);           \
        if (e != hipSuccess) return (int)e;                                                                                   \
        fattn_launch((fattn_relpos_kernel<D, NW, ADD, F16>), dim3((unsigned)grid), dim3(NW * 64), lds, stream, a);    \
    } while (0)
    if (!a.add)          FR_LAUNCH(false, false);
    else if (a.add_f16)  FR_LAUNCH(true, true);
    else                 FR_LAUNCH(true, false);
#undef FR_LAUNCH
    return (int)hipGetLastError();
}

}  // namespace

bool fattn_relpos_supported(const FattnRelposArgs & a) {
    if (a.D != 64 && a.D != 128) return false;
    if (a.Nq < 1 || a.Nkv < 1 || a.H < 1 || a.B < 1) return false;
    // 32-bit tile indices; the table's rows Nq-1+j-i must exist
    if ((int64_t)a.Nq + a.Nkv > (1 << 24)) return false;
    return true;
}

int fattn_relpos_launch(const FattnRelposArgs & a, hipStream_t stream) {
    if (!fattn_relpos_supported(a)) return (int)hipErrorInvalidValue;
    // Workgroups of 2, 3 or 4 waves (32 queries each): no wider than the queries fill, and of those what prices lowest.
    const int64_t heads = (int64_t)a.H * a.B, cus = a.n_cus > 0 ? a.n_cus : 256;
    const int     most  = (a.Nq + 31) / 32 < 4 ? (a.Nq + 31) / 32 : 4;
    auto groups = [&](int waves) { return (a.Nq + 32 * waves - 1) / (32 * waves) * heads; };
    int best = most < 2 ? 2 : most;
    if (a.D == 128 && best == 4) {
        // 128-wide heads have LDS for one workgroup of 4 waves on a CU or for two of 3, and take what fills the chip in fewer
        // rounds.  A 32-key step was measured to take about 1.8 us with 4 waves on the CU, 1.7 with 3 and 3.0 with two times 3 (8
        // heads: 750 tokens x 8 60 us a call with 3 waves against 92 with 4, 1000 x 4 73 against 60; where both are one round, 120
        // x 8 16.1 against 17.7).
        const int64_t wg3 = groups(3), wg4 = groups(4), rest = wg3 % (2 * cus);
        const int64_t t3 = wg3 / (2 * cus) * 30 + (rest == 0 ? 0 : rest <= cus ? 17 : 30), t4 = (wg4 + cus - 1) / cus * 18;
        if (t3 < t4) best = 3;
    } else if (a.D == 64) {
        // 64-wide heads fit by their registers: 8 waves on a CU, as four workgroups of 2, two of 3 or two of 4.  A round takes
        // what the CU with the most waves takes (1000 tokens, us: 33 with 2 waves, 35 with 3, 39 with 4, 47 with 6, 52 with 8).
        // Over 154 calls of 50 to 1500 tokens x 4 to 512 heads this is 0.3% off the best of the three, 7% at worst; 3 waves
        // for all calls, as it was, is 12.5% off (1000 tokens x 64 heads 61.5 us with 2, 96.5 with 3, 61.3 with 4; 120 x 32
        // 10.9, 12.4, 12.4; 750 x 32 38.3, 35.6, 39.1).
        static const int round_of[5][5] = {{}, {}, {0, 33, 40, 47, 52}, {0, 35, 48}, {0, 39, 51}};      // [waves][workgroups on the CU]
        int64_t least = INT64_MAX;
        for (int w = best; w >= 2; w--) {
            const int64_t fit = w == 2 ? 4 : 2, rest = groups(w) % (fit * cus);
            const int64_t t = groups(w) / (fit * cus) * round_of[w][fit] + round_of[w][(rest + cus - 1) / cus];
            if (t < least) { least = t; best = w; }
        }
    }
    static const char * force = getenv("MI355X_RELPOS_WAVES");            // experiments only
    if (force && atoi(force) >= 2 && atoi(force) <= 4) best = atoi(force);
    switch (best) {
        case 2:  return a.D == 64 ? launch_d<64, 2>(a, stream) : launch_d<128, 2>(a, stream);
        case 3:  return a.D == 64 ? launch_d<64, 3>(a, stream) : launch_d<128, 3>(a, stream);
        default: return a.D == 64 ? launch_d<64, 4>(a, stream) : launch_d<128, 4>(a, stream);
    }
}
