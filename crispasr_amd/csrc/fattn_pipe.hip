// Software-pipelined f16-MFMA tile kernel for prefill / encoder attention on gfx950 (CDNA4, wave64).
//
// The products are those of fattn_mma.hip: v_mfma_f32_32x32x16_f16 in transposed form (S^T = K.Q^T, O^T = V^T.P^T), a
// lane owns one query column, probabilities never leave registers.  What differs is the order.  A wave's work is a chain
// of units - 32 queries x 32 keys - and while the exponentials of unit u run on the vector ALU, the matrix cores work on
// the scores of unit u + 1 and on V^T.P^T of unit u - 1: nothing in a region of the loop waits for anything else in it.
// Matrix and vector instructions of ONE wave do overlap on this chip (16 independent 32x32x16 MFMAs with 2 exponentials
// and a conversion behind each: 299 cycles per 8, 271 for the MFMAs alone, 171 for the exponentials), so a wave alone on
// its SIMD keeps the matrix cores busy too.
//
// What the loop had to be rid of to get there, each measured on the 20 x 64-wide encoder layer: taken branches in the
// common path (about 40 cycles each for a wave alone: the steady-state loop is straight-line code and the rare path lies
// behind it), waits on loads just issued.  Matrix instructions and what reads their results are the compiler's, none of them
// inline assembly: it puts the wait states between the two, and leaves them out around instructions it does not know.
//
// K and V blocks of 32 keys go global -> LDS (16 bytes a lane, chunks XOR-swizzled) into a ring of 4 slots each, one
// barrier per block; what a block's start requests is needed two or three blocks later (8 slots are no faster: a CU's path
// from L2 into LDS gives 53 B/clk from two blocks ahead on).  A request is three instructions: a tensor is a buffer that ends with the
// range's last row, so that nothing has to hold a request back inside it, and K's and V's slots have one number.  With clamped row
// numbers and moving bases a request took six and 6 to 12 scalar ones more a step; together with a wait for LDS reads that the
// compiler could not count across the loop's head (a scalar load was on its way), us a pass, in turn on one box: 6 layers of 8 x 64 x
// 1500 against 1536 with their copies 114.7 -> 111.2, 4 of 20 x 64 x 1500^2 x 4 214.7 -> 212.6; 750 x 8 heads of 128 x 8 under a bias (43.5
// and 43.1) and causal 407 and 2048 behind 2048 (90.7, 133.6) within the spread of the runs: two waves a SIMD fill these gaps.  A step's requests go out one
// behind each of its first matrix instructions (a wave alone on its SIMD waits for each to be taken), the last of the prologue's behind
// the first scores: 8 x 64 x 1500 against 1536, K and V from memory, 12.9 -> 12.5 us a launch.
//
// KSP = W: each wave takes two blocks of queries, all that its workgroup has, and every fourth block of keys, which it fetches for itself:
// LDS gives an operand for two products instead of one, and nothing in the loop waits for another wave.  A unit's 0.33 us become 0.27,
// the prologue (its rings are filled by four times as many loads) and the hand-over of four results cost 0.7 us more: 8 x 64 x 1500
// against 1536 12.5 -> 11.75 us a launch, 6 layers with their copies 104 -> 98.
//
// Waves that share queries (KSP > 1) get them through LDS: the workgroup's rows are brought once, along the rows.  A wave's own loads
// of its operands, 32 rows an instruction, took 1.1 us for each 32 queries.  Launches, us, with their own loads and like this: 8 x 64 x
// 1500 against 1536 13.4 -> 12.6, 8 x 64 x 300^2 6.9 -> 6.4; whole passes with both changes, in turn with the code before them: 6 of the
// first layers 111.2 -> 104, four causal layers of 407 tokens, 32 heads of 128, with their row writes 90.8 -> 80.6.  (Eight waves of
// their own 64 queries each: 216.9 and 218.3 us, memory gives the rows no faster.)
//
// Against the tile-wise kernel it replaced for these forms, per launch: 20 x 64 x 1500^2 in batches of 4 60.2 -> 56.8 us
// (0.81 PFLOP/s), 8 x 64 x 1500 against 1536 keys 14.4 -> 12.8, 8 x 128 x 1500^2 x 4 55.2 -> 52.6, 10 x 128 x 1500^2 31.2 ->
// 23.6, 64 x 128 x 300^2 14.9 -> 12.5, 30 x 64 x 300^2 8.8 -> 7.7.
// Workgroups of eight waves, twice the queries (W = 8), bring a CU every block of K and V once instead of twice: the requests,
// timed without them, were 12% of the first of these launches and 15% of the third.  Taken where they fill the CUs as evenly:
// 20 x 64 x 1500^2 x 4 60.6 -> 59.4 us (one box), 12 x 64 x 1500^2 x 4 46.4 -> 42.9, 20 x 64 x 1000^2 x 4 37.2 -> 35.4, 8 x 128 x
// 1500^2 x 4 55.8 -> 53.4, 8 x 128 x 750^2 x 8 33.6 -> 32.0; where they leave more CUs empty they lose (10 x 128 x 1500^2 x 2
// 37.2 -> 44.6).  Eight waves that share the queries of two or four (the keys in turn), for a grid that leaves CUs to one
// workgroup of four, changed nothing at 1500 keys (8 x 64 16.0 us either way) and lost 1 us below 1000.
// Masked calls of 128-wide heads: a wave brings the mask of its next two blocks to LDS as it does K and V, so that the waits
// go on counting, and adds it ahead of the exponentials; the last block may be partial, its keys behind the range excluded by their number.
// Against the tile kernel, whole calls: 2048 causal tokens behind 2048, 32 query and 8 KV heads, with their row writes 146.8 -> 133.4 us, 1000 causal
// tokens 42.5 -> 37.5, 407 (rows that start between dwords, the pairs' form) 21.4 -> 20.1 (now 17.6); under per-head masks 750 x 8 heads x 8
// 45.7 -> 38.8, 1000 x 8 x 4 38.1 -> 32.7, 751 x 8 22.0 -> 19.2.  A step of the 407-token launch is 0.65 us, 32 KB through a CU's
// port; the hand-over and the stores are 3 us of it.
// Hidden keys: the walk ends behind the last 64 that a query of the workgroup sees, starts at the first ones (ranges of 12 tiles and
// more, where that leaves out four), and between the two a hidden block is walked like a visible one - the pairs' form is bound by
// its K and V bytes, which the tile kernel, which skips the block's products, fetches as well.  A row that has seen nothing yet
// stands on a reference below every score: while it stood on -inf its sums were NaN and the wave took the rare path in every step.
// us a call, tile kernel / on -inf and from the first key on / as it is, 8 heads: 1000 causal tokens in a window of 256 21.4 / 24.4 /
// 17.7, four sequences in 900 tokens 20.9 / 24.4 / 16.7, 768 tokens whose first half is hidden 19.0 / 19.0 / 14.6, 500 causal tokens x 4
// padded on the left 16.8 / 18.1 / 16.3, 407 tokens in four sequences (odd rows) 15.5 / 17.3 / 15.3, the middle half of 2048 hidden
// 45.7 / 32.3 / 32.8; 32 heads, 1024 tokens in a window of 256 40.9 / 35.9 / 23.1.  Where no key is hidden ahead of the first: 2048 x 8
// heads, all visible 34.3 -> 34.9 (runs differ by 2%), 1024 x 32 30.1 -> 30.0, causal 29.6 -> 28.6, 407 x 32 16.2 -> 15.75.
// What is left above the MFMAs of a wave alone on its SIMD is not known: its instructions take about 5 cycles each, but a second wave
// that takes half of them changed nothing (above).  Where two
// share a SIMD nothing is full: by the counters of the first of these launches the matrix cores are busy for 49% of it (at
// 1.85 GHz) and the vector ALU for 38%, and a wave stands ready for another instruction to end for 39% of its cycles and
// waits at a counter or barrier for 21%.
#include "fattn_row.h"

#include <type_traits>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float    float16v __attribute__((ext_vector_type(16)));
typedef float    float4v __attribute__((ext_vector_type(4)));
typedef short    short4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

constexpr int   RING         = 4;                  // slots per tensor (a power of two)
constexpr float LOG2E        = 1.4426950408889634f;

template <int D> __device__ __forceinline__ int pipe_swz_k(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
// (for a 32-lane half of a transposing read, rows 0 .. 3, to fall into distinct banks: 64-wide rows lie two to a bank line)
template <int D> __device__ __forceinline__ int pipe_swz_v(int r) { return D == 64 ? ((r >> 1) & 1) << 2 : (r & 3) << 2; }

// LDS by number: a kernel without static LDS finds its dynamic LDS at 0
typedef __attribute__((address_space(3))) const half8 lds_half8;
typedef __attribute__((address_space(3))) short4v     lds_short4;

// instructions stay on their side of it
#define PIPE_FENCE() __builtin_amdgcn_sched_barrier(0)

// A wave's mask block: 32 queries x 32 keys of f16, and for rows that start between dwords the one behind each row's last
constexpr int pipe_mask_slot(int MASK) { return MASK == 2 ? 32 * 64 + 256 : MASK ? 32 * 64 : 0; }
constexpr int pipe_lds_bytes(int D, int NQB, int KSP, int W, int MASK) {
    const int ring  = 2 * RING * KSP * 32 * D * 2 + W * 2 * pipe_mask_slot(MASK) + (MASK && KSP > 1 ? 2 * W * 4 : 0);
    const int stage = W * 32 * D * 4;                                           // result rows / the waves' partial results
    return ring > stage ? ring : stage;
}

// NQB: 32-query blocks per wave.  KSP = 2: the second half of the W waves shares the queries of the first and takes alternate
// 32-key blocks.  KSP = W: see above.
// PAD: heads of a.Dv elements (a multiple of 8 below D) on copies of K and V whose rows are zero-padded to D.
// MASK: 1 where rows start on dwords and Nkv is even, 2 where not; 128-wide heads, no slopes.
template <int D, int NQB, int KSP, int W, bool PAD, int MASK>
__global__ void __launch_bounds__(W * 64, 2) fattn_pipe_kernel(const FattnArgs a, const int n_qtiles) {
    static_assert(NQB == 1 || (NQB == 2 && D == 64 && (KSP == 1 || KSP == W) && !PAD && !MASK), "forms");
    static_assert(!MASK || (D == 128 && NQB == 1 && W == 4 && !PAD), "masked forms");       // (none of them HALVES)
    constexpr int PIPE_THREADS = W * 64;
    constexpr int QG   = W / KSP;                                 // waves that take different queries
    constexpr int KS   = D / 16;                                  // reduction steps of Q.K^T
    constexpr int DB   = D / 32;                                  // 32-wide blocks of the output's d
    constexpr int CH   = D / 8;                                   // 16-byte chunks per row
    constexpr int ROWB = D * 2;
    constexpr int BLKB = 32 * ROWB;                               // bytes of a block
    constexpr int STEPB = KSP * BLKB;                             // ... of a step: one block for every wave of a pair
    constexpr int SKEYS = KSP * 32;
    // A step of one tensor is STEPB / 1024 load instructions.  Every wave makes its share of K's and of V's, NLD each, or (HALVES,
    // where there are fewer of them than waves) the first half of the waves K's and the second V's.
    constexpr bool HALVES = STEPB / 1024 < W;
    constexpr int  NLD  = HALVES ? STEPB / 512 / W : STEPB / 1024 / W;
    constexpr int  NLS  = HALVES ? NLD : 2 * NLD;                 // loads per wave and step
    constexpr int R    = RING;
    // steps ahead of the current one that its start requests, and loads that may still be under way then
    constexpr bool ALONE = KSP == W;                              // a wave fetches the blocks it takes, all of them, and nobody else reads them
    constexpr int DK   = ALONE ? R - 1 : R, DV = NQB == 2 ? DK - 1 : DK - 2;
    constexpr int NML  = MASK == 2 ? 3 : MASK ? 2 : 0;            // ... of its own mask block
    constexpr int AHEAD = DK - 1;                                 // ... of which the last go out behind the first scores
    constexpr int OPEN = (DV - 1) * (NLS + NML);
    constexpr int BMW  = 32 * NQB;
    constexpr int BMG  = BMW * QG;
    constexpr int NM   = KS + 2 * DB;                             // MFMAs of a region
    constexpr int EPS  = 16 / NM;                                 // exponentials per MFMA
    // The reference m enters the scores as the C operand of their first MFMA, 16 registers of one value, and the exponentials
    // need no subtraction.  128-wide heads have vector instructions to spare and no registers: they subtract.
    constexpr bool SPLAT = D == 64;
    // Slot s of the ring holds the K of steps s, s + R, ... and the V of the steps DK - DV before: what a step's start requests goes into one slot
    constexpr uint32_t VRING = R * STEPB, RMASK = R * STEPB - 1;
    auto k_slot = [](uint32_t cur, int ahead) __attribute__((always_inline)) { return (cur + (uint32_t)(ahead + R) * STEPB) & RMASK; };
    auto v_slot = [](uint32_t cur, int ahead) __attribute__((always_inline)) { return (cur + (uint32_t)(ahead + R + DK - DV) * STEPB) & RMASK; };

    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int tid  = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int l32  = lane & 31;
    const int hh   = lane >> 5;
    const int qgroup = wave % QG;
    const int kgroup = wave / QG;

    // Workgroups go to the 8 XCDs round-robin; renumbered so that the query tiles of one (head, batch), which share K/V, sit
    // on one XCD and meet in its L2.
    int bid = blockIdx.x;
    const int nb = gridDim.x, per = nb / 8;
    if (bid < per * 8) bid = (bid % 8) * per + bid / 8;
    const int split = bid % a.n_splits;
    bid /= a.n_splits;
    const int k_begin = split * a.keys_per_split;
    const int k_end   = min(a.Nkv, k_begin + a.keys_per_split);
    int qt = bid % n_qtiles, pair = bid / n_qtiles;
    if (MASK && a.n_splits == 1 && per * 8 == nb && per % n_qtiles == 0) masked_order(per, n_qtiles, a.n_cus, qt, pair);
    // (masked: the batch runs faster than the head, or the longest sequence of a padded batch would be one XCD's alone)
    const int h  = MASK ? pair / a.B : pair % a.Hq;
    const int b  = MASK ? pair % a.B : pair / a.Hq;
    const int hk = h / a.gqa;
    const int bk = b / a.bq;
    const int q0 = qt * BMG + qgroup * BMW;

    // ---- Q rows: requested first, converted behind the first requests of K and V, so that all of them are one round trip ---
    // Where waves share queries the workgroup brings its 64 rows once, to LDS as they are, 16 bytes a lane along the rows (chunks
    // XOR-swizzled), into slots of V's ring that nothing is requested into yet.
    constexpr bool     QLDS  = KSP > 1;
    constexpr int      QCH   = D / 4;                             // 16-byte chunks of a row
    constexpr int      NQL   = BMG * QCH / PIPE_THREADS;          // ... of a lane
    constexpr uint32_t QAT   = VRING;
    static_assert(!QLDS || BMG * D * 4 <= (DK - DV) * STEPB, "the slots ahead of the first V");
    float4v qraw[NQB][QLDS ? 1 : KS][2];
    if constexpr (QLDS) {
        const uint64_t q64  = (uint64_t)(a.q + (int64_t)(qt * BMG) * a.nbq1 + (int64_t)h * a.nbq2 + (int64_t)b * a.nbq3);
        const int      rows = min(BMG, a.Nq - qt * BMG) - 1;
#pragma unroll
        for (int i = 0; i < NQL; i++) {
            const int L = (wave * NQL + i) * 64 + lane, row = L / QCH, c = (L % QCH) ^ (row & 15);
            // (padded: a lane with nothing behind Dv reads the row's first chunk, and its values are scaled by zero)
            load_to_lds16<(MASK != 0)>(q64, (uint32_t)min(row, rows) * (uint32_t)a.nbq1 + (!PAD || c * 4 < a.Dv ? c * 16 : 0), QAT + (wave * NQL + i) * 1024);
        }
    }
#pragma unroll
    for (int qb = 0; qb < (QLDS ? 0 : NQB); qb++) {
        const int qi = min(q0 + qb * 32 + l32, a.Nq - 1);
        const float * qrow = (const float *)(a.q + (int64_t)qi * a.nbq1 + (int64_t)h * a.nbq2 + (int64_t)b * a.nbq3);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            // (padded: a lane with nothing behind Dv reads the row's first 8 elements and scales them by zero)
            const float * q8 = qrow + (!PAD || ks * 16 + hh * 8 < a.Dv ? ks * 16 + hh * 8 : 0);
            qraw[qb][QLDS ? 0 : ks][0] = *(const float4v *)q8;
            qraw[qb][QLDS ? 0 : ks][1] = *(const float4v *)(q8 + 4);
        }
    }

    const int n_keys  = k_end - k_begin;
    int       n_steps = ALONE ? ((n_keys + 31) / 32 + KSP - 1 - kgroup) / KSP : (n_keys + SKEYS - 1) / SKEYS;      // (ALONE: the wave's own, 0 at worst)
    const uint64_t kbase = (uint64_t)(a.k + (int64_t)hk * a.nbk2 + (int64_t)bk * a.nbk3 + (int64_t)k_begin * a.nbk1);
    const uint64_t vbase = (uint64_t)(a.v + (int64_t)hk * a.nbv2 + (int64_t)bk * a.nbv3 + (int64_t)k_begin * a.nbv1);

    // ---- global -> LDS: slot L = (wave * NLD + j) * 64 + lane of a step holds chunk (L % CH) ^ swizzle of row L / CH ------
    // Each tensor is a buffer that ends with the range's last row, each request's address one register that a step moves on: what is
    // requested behind the end is zeros and reaches no memory (its scores are excluded, or nobody looks), and the waits can count.
    const int      lwave = HALVES ? wave % (W / 2) : wave;
    const bool     ofv   = HALVES && wave >= W / 2;               // a wave that loads V alone
    const uint32_t nb1v = (uint32_t)a.nbv1, nb1k = ofv ? nb1v : (uint32_t)a.nbk1;          // (below 2^24)
    const uint32_t inck = SKEYS * nb1k, incv = SKEYS * nb1v;
    const auto     kbuf = fattn_buffer((const void *)(ofv ? vbase : kbase), (uint32_t)(n_keys - 1) * nb1k + ROWB);       // (below 2^31)
    const auto     vbuf = fattn_buffer((const void *)vbase, (uint32_t)(n_keys - 1) * nb1v + ROWB);
    uint32_t kof[NLD], vof[NLD];                                  // (of the request before the next one)
    auto start_at = [&](uint32_t key) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NLD; j++) {
            const int L = (lwave * NLD + j) * 64 + lane, c = L % CH, row = L / CH;
            const uint32_t ck = (uint32_t)((c ^ pipe_swz_k<D>(row & 31)) * 16), cv = (uint32_t)((c ^ pipe_swz_v<D>(row & 31)) * 16);
            kof[j] = __umul24((uint32_t)row, nb1k) + (ofv ? cv : ck) + key * nb1k - inck;
            vof[j] = __umul24((uint32_t)row, nb1v) + cv + key * nb1v - incv;
        }
    };
    start_at(0);
    uint32_t lds0[NLD];
#pragma unroll
    for (int j = 0; j < NLD; j++) lds0[j] = (lwave * NLD + j) * 1024 + (ofv ? VRING : 0);
    auto request_k = [&](uint32_t slot) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NLD; j++) buffer_to_lds16(kbuf, kof[j], inck, lds0[j], slot);
    };
    auto request_v = [&](uint32_t slot) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NLD; j++) buffer_to_lds16(vbuf, vof[j], incv, lds0[j] + VRING, slot);
    };
    // request i < NLS of a step: K's DK steps ahead, V's DV
    auto request_step = [&](uint32_t slot, int i) __attribute__((always_inline)) {
        if (i < NLD) buffer_to_lds16(kbuf, kof[i], inck, lds0[i], slot);
        else         buffer_to_lds16(vbuf, vof[i - NLD], incv, lds0[i - NLD] + VRING, slot);
    };
    // ... and ahead of the first step, as if of the steps before it (a wave that loads V alone leaves out the first DK - DV)
    auto request_first = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int j = from; j < to; j++) {
            if constexpr (HALVES) {
                if (!ofv || j >= DK - DV) request_k(j * STEPB);
            } else {
                request_k(j * STEPB);
                if (j >= DK - DV) request_v(j * STEPB);
            }
        }
    };

    // Operand reads inside this wave's block of a slot: the address of reduction step 0 (of d block 0); step ks (block db) is
    // that with 2 ks (4 db) XORed into the chunk index, which the swizzle passes through.
    const uint32_t kaddr = (uint32_t)((l32 * CH + (hh ^ pipe_swz_k<D>(l32))) * 16 + kgroup * BLKB);
    uint32_t vaddr;
    {
        const int i16 = lane & 15;
        const int kr0 = hh * 4 + (i16 >> 2);
        const int c = ((lane >> 4) & 1) * 2 + ((i16 & 3) >> 1);
        vaddr = (uint32_t)((kr0 * CH + (c ^ pipe_swz_v<D>(kr0))) * 16 + 8 * (i16 & 1) + VRING + kgroup * BLKB);
    }
    // ---- the mask: 32 rows of 64 bytes a block, their 16-byte chunks XOR-swizzled by row, two blocks per wave -----------------
    constexpr uint32_t MSLOT = pipe_mask_slot(MASK);
    const uint32_t m_lds = 2 * R * STEPB + wave * (2 * MSLOT);
    const char * const plane = MASK ? a.mask + (int64_t)(h % a.Hm) * a.nbm2 + (int64_t)(b % a.Bm) * a.nbm3 : nullptr;
    auto row_at = [&](int r) __attribute__((always_inline)) { return (uint32_t)min(q0 + r, a.Nq - 1) * (uint32_t)a.nbm1; };      // (below 2^31)
    // (Rows that start between dwords: from the dword that holds the block's first key on, and the one that holds its last.  Of the mask's
    //  first and last row that can be the two bytes ahead of its first element or behind its last one, in the same dword, so in mapped
    //  memory; they are shifted out.)
    const uint32_t m_odd = MASK == 2 ? (uint32_t)(uint64_t)plane & 2 : 0;
    const auto     mbuf  = fattn_buffer(plane - m_odd, MASK ? (m_odd + (uint32_t)(a.Nq - 1) * (uint32_t)a.nbm1 + (uint32_t)a.Nkv * 2 + 3) & ~3u : 0u);
    uint32_t       mof[MASK ? 3 : 1], m_shift = 0;                // (m_shift: bits from a row's first dword to the block's first key)
    auto start_mask_at = [&](int key) __attribute__((always_inline)) {
        if constexpr (MASK != 0) {
            const uint32_t at = m_odd + (uint32_t)(k_begin + 32 * kgroup + key) * 2;
#pragma unroll
            for (int j = 0; j < 2; j++)
                mof[j] = ((at + row_at(j * 16 + (lane >> 2))) & ~3u) + (uint32_t)(((lane & 3) ^ ((lane >> 4) & 3)) * 16) - SKEYS * 2;
            mof[2]  = MASK == 2 ? ((at + row_at(l32) + 62) & ~3u) - SKEYS * 2 : 0;
            m_shift = MASK == 2 ? ((at + row_at(l32)) & 2) * 8 : 0;
        }
    };
    start_mask_at(0);
    auto request_mask = [&](int slot) __attribute__((always_inline)) {
        if constexpr (MASK != 0) {
#pragma unroll
            for (int j = 0; j < 2; j++) buffer_to_lds16(mbuf, mof[j], SKEYS * 2, m_lds + (slot * MSLOT + j * 1024), 0);
            if (MASK == 2) buffer_to_lds4(mbuf, mof[2], SKEYS * 2, m_lds + (slot * MSLOT + 2048), 0);
        }
    };
    // adds the block in `slot` to scores x of block `block` in log2 units and excludes keys past the end
    auto add_mask = [&](float16v & x, int slot, int block) __attribute__((always_inline)) {
        const uint32_t at = m_lds + slot * MSLOT + (uint32_t)(l32 * 64 + ((l32 >> 2) & 3) * 16);
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) const u32x2 lds_u2;
        typedef __attribute__((address_space(3))) const uint32_t lds_u1;
        u32x2 w[4];
#pragma unroll
        for (int g = 0; g < 4; g++) w[g] = *(lds_u2 *)(uintptr_t)((at ^ (uint32_t)(g * 16)) + 8 * hh);
        if constexpr (MASK == 2) {
            uint32_t next[4];                                     // the dword behind each
#pragma unroll
            for (int g = 0; g < 4; g++)
                next[g] = *(lds_u1 *)(uintptr_t)(hh ? (g < 3 ? at ^ (uint32_t)((g + 1) * 16) : m_lds + slot * MSLOT + 2048 + l32 * 4)
                                                    : (at ^ (uint32_t)(g * 16)) + 8);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                w[g][0] = __builtin_amdgcn_alignbit(w[g][1], w[g][0], m_shift);
                w[g][1] = __builtin_amdgcn_alignbit(next[g], w[g][1], m_shift);
            }
        }
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                x[4 * g + c] = fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(w[g][c >> 1] >> (16 * (c & 1)))), LOG2E, x[4 * g + c]);
        if (__builtin_expect(32 * block + 32 > n_keys, 0)) {
            int lim = n_keys - 32 * block - hh * 4;
            asm volatile("" : "+v"(lim));            // (nothing of this is worth a register in the loop)
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = (r >> 2) * 8 + (r & 3) < lim ? x[r] : -INFINITY;
        }
    };
    // A wave looks at the last 64 keys of its last 8 queries with the first requests; if none of them is seen, at the rows of all its
    // queries, 256 keys at a time from the end on, until it meets a visible key: what lies behind is not walked.  Requests stay
    // inside the rows by moving the last ones back: at worst a block is kept because the one before it is seen.  The first 64 keys
    // of its first 8 queries tell it likewise whether to look for the first key that one of them sees (`first_tile`, below).
    typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
    const int n_tiles = (n_keys + 63) / 64;
    auto mask_keys = [&](int r, int key) __attribute__((always_inline)) {
        return *(const u32x4_a2 *)(plane + (row_at(r) + (uint32_t)min(k_begin + key, k_end - 8) * 2));      // (below 2^32)
    };
    auto any_seen = [&](const u32x4_a2 & w) __attribute__((always_inline)) {                   // (0xFC00: a masked-out key)
        return (w[0] ^ 0xFC00FC00u) | (w[1] ^ 0xFC00FC00u) | (w[2] ^ 0xFC00FC00u) | (w[3] ^ 0xFC00FC00u);
    };
    u32x4_a2 end_keys = {0u, 0u, 0u, 0u}, first_keys = {0u, 0u, 0u, 0u};
    // (the look at the first keys costs 0.4 us where they are visible; below 12 tiles that is what it could save: 640 tokens x 8 heads,
    //  all visible 15.2 us without it and 15.6 with it, in four sequences 15.9 and 14.9)
    const bool from_first = MASK && n_tiles >= 12;
    if constexpr (MASK != 0) {
        end_keys = mask_keys(24 + (lane >> 3), (n_tiles - 1) * 64 + (lane & 7) * 8);
        if (from_first) first_keys = mask_keys(lane >> 3, (lane & 7) * 8);
        request_mask(0);
        request_mask(1);
    }
    request_first(0, AHEAD);

    half8 qreg[NQB][KS];                       // f16 B operands in log2 units
    if constexpr (QLDS) {
        // (the loads behind Q's and the looks at the mask)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NML + (2 * AHEAD - (DK - DV)) * NLD) : "memory");
        __builtin_amdgcn_s_barrier();
    }
#pragma unroll
    for (int qb = 0; qb < NQB; qb++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            float4v x[2];
            if constexpr (QLDS) {
                typedef __attribute__((address_space(3))) const float4v lds_float4;
                const int row = (qgroup * NQB + qb) * 32 + l32;
#pragma unroll
                for (int e = 0; e < 2; e++) x[e] = *(lds_float4 *)(uintptr_t)(QAT + row * (D * 4) + (((ks * 4 + hh * 2 + e) ^ (row & 15)) * 16));
            } else {
                asm volatile("" : "+v"(qraw[qb][QLDS ? 0 : ks][0]), "+v"(qraw[qb][QLDS ? 0 : ks][1]));          // (not before here)
                x[0] = qraw[qb][QLDS ? 0 : ks][0];
                x[1] = qraw[qb][QLDS ? 0 : ks][1];
            }
            const float qs = !PAD || ks * 16 + hh * 8 < a.Dv ? a.scale * LOG2E : 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) qreg[qb][ks][e] = (_Float16)(x[e >> 2][e & 3] * qs);
        }

    // (in the slot of V's that the first region asks for, or behind the masks where Q is in that; read behind the barrier below)
    int * const ends = (int *)(lds + (QLDS ? 2 * R * STEPB + W * 2 * MSLOT : VRING + v_slot(0, DV)));
    if constexpr (MASK != 0) {
        int  nt = n_tiles, ft = 0, at = 0;                       // at: tiles looked at from the end in question
        bool last  = __builtin_amdgcn_ballot_w64(any_seen(end_keys) != 0) == 0;
        bool first = from_first && __builtin_amdgcn_ballot_w64(any_seen(first_keys) != 0) == 0;
        // (One loop for both ends, the last one first, in line: a launch behind other kernels fetches the code anew, and what lies out of
        //  line costs a jump to it.  Four layers of 407 tokens with their row writes and conversions, the same inputs each pass: 91.0 us
        //  with the look at the end alone, 94 with two loops or with this one out of line, 91.5 like this; five inputs in turn 100 and 96.)
        if (last || first) {
#pragma unroll 1
            do {
                const int hi = n_tiles - at, lo = last ? max(hi - 4, 0) : at;
                u32x4_a2  w[16 / KSP];             // (the two waves of a pair share the rows)
                uint32_t  any = 0;
#pragma unroll
                for (int i = 0; i < 16 / KSP; i++) w[i] = mask_keys(kgroup * 16 + i * 2 + (lane >> 5), lo * 64 + (lane & 31) * 8);
#pragma unroll
                for (int i = 0; i < 16 / KSP; i++) any |= any_seen(w[i]);
                asm volatile("" : "+v"(any));      // (one word: else the compiler keeps 32 compares' results in scalar registers)
                const uint64_t v2 = __builtin_amdgcn_ballot_w64(any != 0);
                const uint32_t v  = (uint32_t)v2 | (uint32_t)(v2 >> 32);        // runs of 8 keys
                if (v == 0 && (last ? hi > 4 : at + 4 < nt)) {
                    at += 4;
                } else if (last) {
                    nt   = v ? min(hi, lo + (31 - __builtin_clz(v)) / 8 + 1) : 1;
                    last = false;
                    at   = 0;
                } else {
                    ft    = v ? lo + __builtin_ctz(v) / 8 : nt;
                    first = false;
                }
            } while (last || first);
        }
        if (lane == 0) {
            ends[wave]     = nt;
            ends[W + wave] = ft;
        }
    }

    float16v oacc[NQB][DB], negm[SPLAT ? NQB : 1], s[2];
    half8    p[2][2];
    float    m[NQB];
    float4v  lacc[NQB];                       // row sums: four times the same number
#pragma unroll
    for (int qb = 0; qb < NQB; qb++) {
        lacc[qb] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[qb][db][r] = 0.0f;
    }
    half8 zero8;
#pragma unroll
    for (int e = 0; e < 8; e++) zero8[e] = (_Float16)0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int k = 0; k < 2; k++) p[i][k] = zero8;
    // Row sums by the matrix cores: row i of this constant operand of v_mfma_f32_16x16x32_f16 has ones where
    // (i / 4) % 2 == (k / 8) % 2, so that every lane finds in its accumulators the sum of the probabilities that it and
    // the lane 32 away supply for their query - the rounded ones that V is multiplied by.
    half8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (_Float16)(((lane >> 2) & 1) == ((lane >> 4) & 1) ? 1.0f : 0.0f);

    // Operand registers.  Two query blocks per wave: K of one block, V of one block, each used twice.  One query block: two
    // sets of 4 MFMA operands, Y and X, that take turns - 128-wide heads: the first and second half of K, then of V.
    constexpr bool TURNS = NQB == 1 && D == 128;
    half8 ka[TURNS ? 4 : KS], va[TURNS ? 4 : 2 * DB];             // TURNS: Y = ka, X = va
#pragma unroll
    for (int i = 0; i < (TURNS ? 4 : 2 * DB); i++) va[i] = zero8;
    auto read_k = [&](half8 (&to)[4], uint32_t slot, int ks0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) to[i] = *(lds_half8 *)(uintptr_t)((slot + kaddr) ^ (uint32_t)((ks0 + i) * 32));
    };
    auto read_v1 = [&](uint32_t slot, int k2, int db) __attribute__((always_inline)) {
        lds_short4 * p0 = (lds_short4 *)(uintptr_t)(((slot + vaddr) ^ (uint32_t)(db * 64)) + k2 * 16 * ROWB);
        const half4 lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(p0));
        const half4 hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(p0 + ROWB));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto read_v = [&](half8 (&to)[4], uint32_t slot, int i0) __attribute__((always_inline)) {      // operands i0 .. i0 + 3 of (k2, db)
#pragma unroll
        for (int i = 0; i < 4; i++) to[i] = read_v1(slot, (i0 + i) / DB, (i0 + i) % DB);
    };

    // the first two blocks of K have landed
    auto first_landed = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(HALVES ? (AHEAD - 2) * NLD : (2 * AHEAD - 2 - (DK - DV)) * NLD) : "memory");
        __builtin_amdgcn_s_barrier();
    };
    auto clear_first_v = [&]() __attribute__((always_inline)) {
        // the first unit multiplies the V of a step before the first one by zeros: it must be finite
#pragma unroll
        for (int i = 0; i < STEPB / 16 / PIPE_THREADS; i++) *(float4 *)(lds + VRING + v_slot(0, -1) + (i * PIPE_THREADS + tid) * 16) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    };
    if (NQB == 1 && !QLDS) clear_first_v();
    first_landed();
    if (NQB == 1 && QLDS) clear_first_v();             // (every wave has read Q there)
    int first_step = 0;
    if constexpr (MASK != 0) {
        n_steps = min(n_steps, max(max(ends[0], ends[1]), max(ends[2], ends[3])) * 64 / SKEYS);
        // Keys that no query of the workgroup sees before the first one (windows, padding on the left, several sequences in a row):
        // the requests start again behind them, where that leaves out four tiles or more (2.6 us for 1.5).
        const int first_tile = __builtin_amdgcn_readfirstlane(min(min(ends[W], ends[W + 1]), min(ends[W + 2], ends[W + 3])));
        if (first_tile >= 4 && first_tile * 64 / SKEYS < n_steps) {
            first_step = first_tile * 64 / SKEYS;
            // every wave has read `ends`, and nothing is on its way into the slots
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            start_at((uint32_t)first_tile * 64);
            start_mask_at(first_tile * 64);
            request_mask(0);
            request_mask(1);
            request_first(0, AHEAD);
            first_landed();
        }
    }
    auto exclude_past_end = [&](float16v & x, int step) __attribute__((always_inline)) {
        int lim = n_keys - step * SKEYS - kgroup * 32 - hh * 4;
        asm volatile("" : "+v"(lim));            // (nothing of this is worth a register in the loop)
#pragma unroll
        for (int r = 0; r < 16; r++) x[r] = (r >> 2) * 8 + (r & 3) < lim ? x[r] : -INFINITY;
    };
    // the first reference of every row: its largest score in the first block
    {
        half8 k1[4];
        read_k(ka, 0, 0);
        if (KS == 8) read_k(k1, 0, KS - 4);
#pragma unroll
        for (int qb = NQB - 1; qb >= 0; qb--) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[0][r] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ks < 4 ? ka[ks & 3] : k1[ks & 3], qreg[qb][ks], s[0], 0, 0, 0);
            float16v first = s[0];
            if constexpr (MASK != 0)  add_mask(first, 0, KSP * first_step + kgroup);       // (its own turn comes with the first region)
            else if (n_keys < SKEYS) { exclude_past_end(s[0], 0); first = s[0]; }
            float mx = first[0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = fmaxf(mx, first[r]);
            mx = max_of_halves(mx);
            // (masked rows that see nothing yet stand below every score: the exponentials of hidden keys are zeros, and the first key
            //  that such a row sees leaves f16's range, so that the rare path below gives it a reference)
            m[qb] = mx > -INFINITY ? mx : MASK ? -3.0e38f : 0.0f;
            if (SPLAT) {
#pragma unroll
                for (int r = 0; r < 16; r++) negm[SPLAT ? qb : 0][r] = -m[qb];
            }
        }
        if (SPLAT) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[0][r] -= m[0];
        }
        if (NQB == 1) read_k(ka, STEPB, 0);      // (of a single step: what the slot holds, multiplied and not used)
    }

    int      step = first_step;
    uint32_t cur  = 0;                                            // slot of the current step

    // One unit: the softmax of s[U] (query block QB), with the scores of the next unit into s[1 - U] and V^T.P^T of the one
    // before on the matrix cores.
    auto region = [&](auto u_tag) __attribute__((always_inline)) {
        constexpr int  U     = decltype(u_tag)::value;
        constexpr bool START = NQB == 1 || U == 0;                // the first unit of a step
        constexpr int  QB    = NQB == 2 ? U : 0, NX = NQB == 2 ? 1 - U : 0;
        if constexpr (START) {
            // what was requested OPEN loads ago and earlier has landed, in every wave's share
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OPEN) : "memory");
            if (!ALONE) __builtin_amdgcn_s_barrier();
        }
        if constexpr (MASK != 0) {
            add_mask(s[U], U, KSP * step + kgroup);
            PIPE_FENCE();
            request_mask(U);
        } else if (__builtin_expect(step * SKEYS > n_keys - 32 * kgroup - 32, 0)) exclude_past_end(s[U], step);
        // (one query block) operands of this region's second half
        if (TURNS)          read_k(va, k_slot(cur, 1), KS - 4);
        else if (NQB == 1)  read_v(va, v_slot(cur, -1), 0);
        PIPE_FENCE();
        float e[16];
        float lprev = lacc[QB][0];                                // (a copy by force: else all four old sums stay in registers)
        asm volatile("" : "+v"(lprev));
        auto pack = [&](int i) __attribute__((always_inline)) {          // probabilities 2i, 2i + 1
            p[U][i >> 2][(2 * i) & 7]     = (_Float16)e[2 * i];
            p[U][i >> 2][(2 * i + 1) & 7] = (_Float16)e[2 * i + 1];
        };
        auto add_sums = [&](int k) __attribute__((always_inline)) { lacc[QB] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, p[U][k], lacc[QB], 0, 0, 0); };
        int done = 0, packed = 0;
#pragma unroll
        for (int j = 0; j < NM; j++) {
            // operands that take the place of those that the MFMA before has read for the last time
            if (TURNS && j == 4)                         read_v(ka, v_slot(cur, -1), 0);
            if (TURNS && j == 8)                         read_v(va, v_slot(cur, -1), 4);
            if (TURNS && j == 12)                        read_k(ka, k_slot(cur, 2), 0);
            if (!TURNS && NQB == 1 && j == KS)           read_k(ka, k_slot(cur, 2), 0);
            if (NQB == 2 && U == 0 && j == KS)           read_k(ka, k_slot(cur, 1), 0);
            PIPE_FENCE();
            if (j == 0) {
                if (SPLAT) {
                    s[1 - U] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[0], qreg[NX][0], negm[SPLAT ? NX : 0], 0, 0, 0);
                } else {
                    float16v none;
#pragma unroll
                    for (int r = 0; r < 16; r++) none[r] = 0.0f;
                    s[1 - U] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[0], qreg[NX][0], none, 0, 0, 0);
                }
            }
            else if (j < KS)  s[1 - U] = __builtin_amdgcn_mfma_f32_32x32x16_f16(TURNS && j >= 4 ? va[j & 3] : ka[j & 3], qreg[NX][j], s[1 - U], 0, 0, 0);
            else {
                const int i = j - KS, k2 = i / DB, db = i % DB;
                oacc[NX][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(TURNS ? (k2 ? va[db & 3] : ka[db & 3]) : va[i % (2 * DB)], p[1 - U][k2], oacc[NX][db], 0, 0, 0);
            }
            if (START && j < NLS) request_step(k_slot(cur, DK), j);
#pragma unroll
            for (int k = 0; k < EPS; k++) { e[done] = __builtin_amdgcn_exp2f(SPLAT ? s[U][done] : s[U][done] - m[QB]); done++; }
            while (packed * 2 + 2 <= done - EPS) { pack(packed); packed++; }
            if (j == NM - 2) add_sums(0);
            PIPE_FENCE();
        }
        if (NQB == 2 && U == 0) read_v(va, v_slot(cur, 0), 0);
#pragma unroll
        for (; packed < 8; packed++) pack(packed);
        add_sums(1);
        if (NQB == 1 || U == 1) cur = k_slot(cur, 1);
        PIPE_FENCE();
        // A probability that left f16's range (inf, or NaN from an infinite score) shows in the row's sum: the reference has
        // fallen 16 binary orders behind.  Wave-uniform and rare.  It shows in the sum of the row 16 away too, which shares columns of
        // `ones` with it: what is still not finite under the raised reference is left out of the sums here and added to its own row's, so
        // that a row of NaN, which comes this way with every unit, leaves the others as they are.  (v_mfma_f32_4x4x4_16b_f16, which mixes
        // no rows, is 2 to 6% slower: 12 x 64 x 1500^2 x 4 40.5 and 43.1 us.)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(lacc[QB][0] <= 1e30f)) != 0, 0)) {
            float mx = s[U][0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[U][r]);
            float delta = 0.0f, f, base;                           // base: what the scores at hand still have to come down by
            if constexpr (MASK != 0) {
                base  = fmaxf(max_of_halves(mx), m[QB]);
                f     = base == m[QB] ? 1.0f : __builtin_amdgcn_exp2f(m[QB] - base);
                m[QB] = base;
            } else {
                delta = fmaxf(max_of_halves(mx) - (SPLAT ? 0.0f : m[QB]), 0.0f);
                f     = __builtin_amdgcn_exp2f(-delta);
                base  = SPLAT ? delta : m[QB] + delta;
                m[QB] += delta;
            }
            if (!MASK || __builtin_amdgcn_ballot_w64(lprev != 0.0f && f != 1.0f) != 0) {       // (not where rows see their first keys)
#pragma unroll
                for (int db = 0; db < DB; db++)
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[QB][db][r] *= f;
            }
            if (SPLAT) {
#pragma unroll
                for (int r = 0; r < 16; r++) negm[SPLAT ? QB : 0][r] -= delta;
                if (NQB == 1) {          // the next unit's scores stand on the old reference
#pragma unroll
                    for (int r = 0; r < 16; r++) s[1 - U][r] -= delta;
                }
            }
            float odd = 0.0f;                                      // 0, or NaN
#pragma unroll
            for (int i = 0; i < 8; i++) {
                e[2 * i]     = __builtin_amdgcn_exp2f(s[U][2 * i] - base);
                e[2 * i + 1] = __builtin_amdgcn_exp2f(s[U][2 * i + 1] - base);
                odd          = fmaf(e[2 * i] + e[2 * i + 1], 0.0f, odd);
                pack(i);
                PIPE_FENCE();
            }
            odd = sum_of_halves(odd);
#pragma unroll
            for (int r = 0; r < 4; r++) lacc[QB][r] = fmaf(lprev, f, odd);
#pragma unroll
            for (int k = 0; k < 2; k++) lacc[QB] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, odd == 0.0f ? p[U][k] : zero8, lacc[QB], 0, 0, 0);
        }
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    // V^T.P^T of the last unit
    auto last_pv = [&](auto u_tag) __attribute__((always_inline)) {
        constexpr int U = decltype(u_tag)::value, QB = NQB == 2 ? U : 0;
#pragma unroll
        for (int k2 = 0; k2 < 2; k2++)
#pragma unroll
            for (int db = 0; db < DB; db++) {
                const half8 v = NQB == 2 ? va[(k2 * DB + db) % (2 * DB)] : read_v1(v_slot(cur, -1), k2, db);
                oacc[QB][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, p[U][k2], oacc[QB][db], 0, 0, 0);
            }
    };
    // (One query block: an odd number of steps is made even by one whose keys all lie past the end.  Leaving the loop in the
    //  middle would cost the accumulators' 64 registers a copy in every turn.)
    request_first(AHEAD, DK);
    __builtin_amdgcn_s_waitcnt(0xC07F);                          // lgkmcnt(0), known to the compiler: scalar loads on their way are not counted
#pragma unroll 1
    while (step < n_steps) {
        region(I0{});
        if (NQB == 1) step++;
        region(I1{});
        step++;
    }
    last_pv(I1{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (what was requested behind the last step)

    __syncthreads();                                   // every wave is done with the ring
    // Excluded keys were multiplied by probabilities of zero, not skipped: the same for finite K/V, NaN otherwise.  Queries whose
    // result is not finite are left out below and computed at the end, excluded keys unread, as the CPU op does it.
    uint32_t bad = 0;                                      // (lanes l and l + 32 hold the same query)
    if constexpr (MASK != 0) {
        float chk = lacc[0][0] * 0.0f;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) chk = fmaf(oacc[0][db][r], 0.0f, chk);
        const uint64_t bits = __builtin_amdgcn_ballot_w64(chk != 0.0f);
        bad = (uint32_t)bits | (uint32_t)(bits >> 32);
    }

    // ---- the two waves of a pair hand each other half of the result's columns through LDS ----------------------------------
    if constexpr (KSP == 2) {
        constexpr int HB    = DB / 2;
        constexpr int XREGS = HB * 16 + 3;                 // accumulators, reference, sum, bad rows: one dword per lane each
        static_assert(W * XREGS * 256 <= pipe_lds_bytes(D, NQB, KSP, W, MASK), "hand-over");
        auto trade = [&](auto first) __attribute__((always_inline)) {
            constexpr int MINE = decltype(first)::value * HB, THEIRS = HB - MINE;
            float * const out = (float *)lds + wave * (XREGS * 64) + lane;
            const float * const in = (const float *)lds + (wave ^ QG) * (XREGS * 64) + lane;
#pragma unroll
            for (int db = 0; db < HB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) out[(db * 16 + r) * 64] = oacc[0][THEIRS + db][r];
            out[(HB * 16) * 64]     = m[0];
            out[(HB * 16 + 1) * 64] = lacc[0][0];
            out[(HB * 16 + 2) * 64] = __uint_as_float(bad);
            __syncthreads();
            // (a wave without a key of its own has a sum of zero)
            const float mo = in[(HB * 16) * 64], lo = in[(HB * 16 + 1) * 64];
            const float mn = lo == 0.0f ? m[0] : lacc[0][0] == 0.0f ? mo : fmaxf(m[0], mo);
            const float fa = lacc[0][0] == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(m[0] - mn);
            const float fo = lo == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(mo - mn);
            lacc[0][0] = lacc[0][0] * fa + lo * fo;
#pragma unroll
            for (int db = 0; db < HB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[0][db][r] = oacc[0][MINE + db][r] * fa + in[(db * 16 + r) * 64] * fo;
            m[0] = mn;
            bad |= (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(in[(HB * 16 + 2) * 64]));
        };
        if (kgroup == 0) trade(I0{});
        else             trade(I1{});
    }

    // ---- ... and the four that have its keys among them: wave 2 qb + db gets block db of the columns of query block qb --------
    float16v part = {};
    if constexpr (ALONE) {
        static_assert(!ALONE || (W == 4 && NQB * DB == W), "a block for every wave");
        static_assert(!ALONE || W * W * 4096 + W * NQB * 512 <= pipe_lds_bytes(D, NQB, KSP, W, MASK), "hand-over");
        float4v * const box = (float4v *)lds + lane;                             // [wave][block][quarter][lane]
        float2 * const  ml  = (float2 *)(lds + W * W * 4096) + lane;             // [wave][query block][lane]
#pragma unroll
        for (int i = 0; i < W; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float16v & o = oacc[i / DB][i % DB];
                box[((wave * W + i) * 4 + g) * 64] = float4v{o[4 * g], o[4 * g + 1], o[4 * g + 2], o[4 * g + 3]};
            }
#pragma unroll
        for (int qb = 0; qb < NQB; qb++) ml[(wave * NQB + qb) * 64] = make_float2(m[qb], lacc[qb][0]);
        __syncthreads();
        // (a wave without a key of its own has a sum of zero)
        float2 of[W];
        float  M = -INFINITY, L = 0.0f;
#pragma unroll
        for (int w = 0; w < W; w++) of[w] = ml[(w * NQB + wave / DB) * 64];
#pragma unroll
        for (int w = 0; w < W; w++) M = of[w].y == 0.0f ? M : fmaxf(M, of[w].x);
#pragma unroll
        for (int w = 0; w < W; w++) {
            const float f = of[w].y == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(of[w].x - M);
            L += of[w].y * f;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4v o = box[((w * W + wave) * 4 + g) * 64];
#pragma unroll
                for (int e = 0; e < 4; e++) part[4 * g + e] += o[e] * f;
            }
        }
        m[0]       = M;
        lacc[0][0] = L;
    }

    // ---- normalise and write dst[D, Hq, Nq, B], or hand the unnormalised partial to the merge kernel -----------------------
    const int dv = PAD ? a.Dv : D;                      // rows of dv floats; the partials' are D apart
    if constexpr (KSP == 1) {
        // whole rows through LDS (32 x D floats per wave, chunks XOR-swizzled by row), 16 or 32 adjacent lanes on one row
        constexpr int CPR = D / 4;                         // 16-byte chunks per output row
        constexpr int RPI = 64 / CPR;                      // rows per store instruction
        float * const stg = (float *)lds + qgroup * (32 * D);
        const int64_t row_stride = a.n_splits > 1 ? (int64_t)a.Hq * a.n_splits * D : (int64_t)a.Hq * dv;    // floats between queries
#pragma unroll
        for (int qb = 0; qb < NQB; qb++) {
            const float ltot = lacc[qb][0];
            const float inv  = a.n_splits > 1 ? 1.0f : (ltot > 0.0f ? 1.0f / ltot : 0.0f);
            const int   qi   = q0 + qb * 32 + l32;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    float4 o;
                    o.x = oacc[qb][db][g * 4 + 0] * inv;
                    o.y = oacc[qb][db][g * 4 + 1] * inv;
                    o.z = oacc[qb][db][g * 4 + 2] * inv;
                    o.w = oacc[qb][db][g * 4 + 3] * inv;
                    const int c = db * 8 + g * 2 + hh;
                    *(float4 *)(stg + l32 * D + ((c ^ (l32 & (CPR - 1))) * 4)) = o;
                }
            __builtin_amdgcn_wave_barrier();               // (LDS serves a wave's requests in order)
            const int     q_first = q0 + qb * 32;
            const int64_t row0    = ((int64_t)b * a.Nq + q_first) * a.Hq + h;
            float * const out0    = a.n_splits > 1 ? a.part_acc + (row0 * a.n_splits + split) * D : a.dst + row0 * dv;
#pragma unroll
            for (int k = 0; k < 32 / RPI; k++) {
                const int row = k * RPI + lane / CPR, c = lane % CPR;
                const float4 o = *(const float4 *)(stg + row * D + ((c ^ (row & (CPR - 1))) * 4));
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                if (q_first + row < a.Nq && (!PAD || c * 4 < a.Dv) && (!MASK || !(bad >> row & 1)))
                    __builtin_nontemporal_store(f32x4{o.x, o.y, o.z, o.w}, (f32x4 *)(out0 + row * row_stride + c * 4));
            }
            __builtin_amdgcn_wave_barrier();               // the next query block reuses the staging rows
            if (a.n_splits > 1 && hh == 0 && qi < a.Nq && (!MASK || !(bad >> l32 & 1))) {
                // (reference, sum) in natural-log units; a range with no visible key contributes nothing
                float * pm = a.part_ml + ((((int64_t)b * a.Nq + qi) * a.Hq + h) * a.n_splits + split) * 2;
                pm[0] = ltot == 0.0f ? -INFINITY : m[qb] * 0.6931471805599453f;
                pm[1] = ltot;
            }
        }
    } else {
        // (short launches: straight from the accumulators, the detour would cost them a round trip)
        const float ltot = lacc[0][0];
        const float inv  = a.n_splits > 1 ? 1.0f : (ltot > 0.0f ? 1.0f / ltot : 0.0f);
        const int   qi   = q0 + (ALONE ? wave / DB * 32 : 0) + l32;
        if (qi < a.Nq && (!MASK || !(bad >> l32 & 1))) {
            const int64_t row = ((int64_t)b * a.Nq + qi) * a.Hq + h;
            float * out = a.n_splits > 1 ? a.part_acc + (row * a.n_splits + split) * D : a.dst + row * dv;
#pragma unroll
            for (int i = 0; i < DB / 2; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float16v & x = ALONE ? part : oacc[0][i];
                    float4 o;
                    o.x = x[g * 4 + 0] * inv;
                    o.y = x[g * 4 + 1] * inv;
                    o.z = x[g * 4 + 2] * inv;
                    o.w = x[g * 4 + 3] * inv;
                    const int d = ((ALONE ? wave % DB : kgroup * (DB / 2)) + i) * 32 + g * 8 + hh * 4;
                    if (!PAD || d < a.Dv) *(float4 *)(out + d) = o;
                }
            if (a.n_splits > 1 && hh == 0 && (ALONE ? wave % DB : kgroup) == 0) {
                float * pm = a.part_ml + (row * a.n_splits + split) * 2;
                pm[0] = ltot == 0.0f ? -INFINITY : m[0] * 0.6931471805599453f;
                pm[1] = ltot;
            }
        }
    }
    if constexpr (MASK != 0) {
        if (bad != 0 && kgroup == 0) {
            for (; bad != 0; bad &= bad - 1) {
                const int qi = q0 + __builtin_ctz(bad);
                if (qi < a.Nq) attn_row_redo<MI355X_TYPE_F16, D>(a, qi, h, b, split, k_begin, k_end);
            }
        }
    }
}

template <int D, int NQB, int KSP, int W, bool PAD, int MASK = 0>
int launch(const FattnArgs & a, hipStream_t stream) {
    constexpr int bmg = 32 * NQB * W / KSP, lds = pipe_lds_bytes(D, NQB, KSP, W, MASK);
    const int     n_qtiles = (a.Nq + bmg - 1) / bmg;
    const int64_t wgs = (int64_t)n_qtiles * a.Hq * a.B * a.n_splits;
    if (wgs > 0x7fffffff) return (int)hipErrorInvalidValue;
    static std::atomic<uint64_t> lds_allowed{0};
    const hipError_t e = fattn_allow_lds((const void *)fattn_pipe_kernel<D, NQB, KSP, W, PAD, MASK>, lds, lds_allowed);
    if (e != hipSuccess) return (int)e;
    fattn_launch((fattn_pipe_kernel<D, NQB, KSP, W, PAD, MASK>), dim3((unsigned)wgs), dim3(W * 64), (size_t)lds, stream, a, n_qtiles);
    return (int)hipGetLastError();
}

}  // namespace

// The masked calls among those over f16 rows: whole 128-wide heads, no slopes.  Rows that start between dwords need LDS that two
// workgroups of the unsplit form do not have on one CU.  Ranges from 64 keys on for pairs of waves, from 128 for the unsplit form (a caller
// who names the form: 384, as ever).  us a call in a graph, tile kernel and this: pairs, four causal layers of 383 tokens x 32 heads with
// their row writes 87.0, 69.9, of 256 66.3, 58.8, of 128 55.1, 51.4, of 100 52.4, 50.5; under per-head masks 100 x 8 heads 10.9, 9.5, 300 x 8
// 14.1, 12.1; unsplit, 150 x 8 heads x 16 16.0, 14.3, 250 x 8 x 16 20.5, 17.4, 380 x 8 x 8 21.3, 17.9.
static bool pipe_masked(const FattnArgs & a, const FattnMmaVariant & v) {
    const int least = a.tile_variant ? 384 : v.key_split == 2 ? 64 : 128;
    return a.D == 128 && a.Dv == 128 && v.query_blocks == 1 && a.max_bias <= 0.0f &&
           (a.n_splits > 1 ? a.keys_per_split : a.Nkv) >= least && (uint64_t)a.Nq * (uint64_t)a.nbm1 < (1ull << 31) &&
           (v.key_split == 2 || (a.mask_al4 && !(a.Nkv & 1)));
}

// The pairs' form of 128-wide heads takes 128 keys a turn and starts with more requests than the tile kernel, whose waves have 64 and are done
// sooner with few rows: those of one tile, or three, stay that kernel's, and all of half a tile.  us a call in a graph, tile kernel and pairs, 8 heads, 9 rows x
// 32 keys 5.4, 6.35, 17 x 64 5.6, 6.25, 48 x 32 6.7, 6.9, x 64 6.7, 6.7, 64 x 32 7.1, 7.05, x 64 7.15, 6.8; 3 x 129 6.7, 7.4, 17 x 160 7.0, 7.3, 24 x 129 7.25, 7.5,
// x 192 7.25, 7.25, 32 x 160 7.55, 7.45; 9 x 100 6.2, 6.05, 9 x 193 7.55, 7.1, 40 heads, 8 x 288 8.35, 8.35; 96-wide 40 x 32 8.45, 8.8.
static bool few_rows_of_odd_tiles(const FattnArgs & a) {
    const int keys = a.n_splits > 1 ? a.keys_per_split : a.Nkv;
    return keys <= 32 || a.Nq <= (keys <= 64 ? 48 : keys > 128 && keys <= 192 ? 24 : 0);
}

// Request addresses are 32-bit numbers inside a range of a head's keys, up to 8 steps of 64 behind its end, and inside the 64 rows of Q that
// waves share: what lies further apart is the tile kernel's.
bool fattn_pipe_reaches(const FattnArgs & a, int64_t keys, bool shared_q) {
    const int64_t lim = (int64_t)1 << 31;
    return (keys + 8 * 64) * a.nbk1 < lim && (keys + 8 * 64) * a.nbv1 < lim && (!shared_q || (a.nbq1 >= 0 && a.nbq1 < 1 << 25));
}

// Plain attention over f16 rows is this kernel's.  (The pairs' form of 128-wide heads since queries come through LDS; us a layer, tile
// kernel and this: 8 heads x 80 7.9, 6.9, x 300 11.0, 9.75, x 1500 25.6, 19.8, 10 x 1000 20.0, 15.45, 80-wide 8 x 1500 31.0, 24.9.)
// Eight waves a workgroup where that leaves no CU with more of them than workgroups of four do: more of those than CUs, and their
// number per CU even once rounded up.  (A caller who names the form gets four.)
int fattn_pipe_waves(const FattnArgs & a, int ktype, const FattnMmaVariant & v) {
    if (ktype != MI355X_TYPE_F16 || !v.direct || a.softcap != 0.0f) return 0;
    if (!fattn_pipe_reaches(a, a.n_splits > 1 ? a.keys_per_split : a.Nkv, v.key_split > 1)) return 0;
    if (a.masked) return pipe_masked(a, v) ? 4 : 0;
    if (v.key_split == 2) return a.D == 128 && few_rows_of_odd_tiles(a) ? 0 : 4;
    if (a.tile_variant != 0 || (a.D == 64 && v.query_blocks != 2)) return 4;
    const int q4 = v.queries_per_workgroup;
    auto groups  = [&](int q) { return (int64_t)((a.Nq + q - 1) / q) * a.Hq * a.B * a.n_splits; };
    auto fill    = [&](int64_t wgs) { return (wgs + a.n_cus - 1) / a.n_cus; };
    return groups(q4) > a.n_cus && 2 * fill(groups(2 * q4)) <= fill(groups(q4)) ? 8 : 4;
}

// Calls of the pairs' form whose four waves rather take different keys of the same 64 queries (KSP = W): a CU holds one such workgroup,
// and its waves have to have keys enough for the longer hand-over.  us a call, pairs and like this, in graphs: 8 heads x 1500 13.2, 12.6,
// x 1000 10.4, 10.1, x 768 8.9, 8.9, x 500 7.4, 7.7; 4 x 1500 12.7, 12.0, 4 x 800 9.7, 9.25.  Nearly every CU with one (all ask L2 for
// their keys at once): 12 x 1300 14.05, 13.5, 16 x 1000 11.5, 11.8.
bool fattn_pipe_alone(const FattnArgs & a, const FattnMmaVariant & v) {
    if (a.masked || a.D != 64 || a.Dv != a.D || v.key_split != 2) return false;
    const int64_t wgs = (int64_t)((a.Nq + 63) / 64) * a.Hq * a.B * a.n_splits;
    return a.tile_variant == 0 && wgs <= a.n_cus && (a.n_splits > 1 ? a.keys_per_split : a.Nkv) >= (wgs * 8 <= (int64_t)a.n_cus * 7 ? 768 : 1152);
}

int fattn_pipe_launch(const FattnArgs & a, const FattnMmaVariant & v, int waves, hipStream_t stream) {
    const bool pad = a.Dv != a.D;
    if (a.masked) {
        const bool dwords = a.mask_al4 && !(a.Nkv & 1);
        if (v.key_split == 2) return dwords ? launch<128, 1, 2, 4, false, 1>(a, stream) : launch<128, 1, 2, 4, false, 2>(a, stream);
        return launch<128, 1, 1, 4, false, 1>(a, stream);
    }
    if (v.query_blocks == 2) {
        if (pad || a.D != 64) return (int)hipErrorInvalidValue;
        return waves == 8 ? launch<64, 2, 1, 8, false>(a, stream) : launch<64, 2, 1, 4, false>(a, stream);
    }
    if (a.D == 64) {
        if (fattn_pipe_alone(a, v)) return launch<64, 2, 4, 4, false>(a, stream);
        if (v.key_split == 2) return pad ? launch<64, 1, 2, 4, true>(a, stream) : launch<64, 1, 2, 4, false>(a, stream);
        return pad ? launch<64, 1, 1, 4, true>(a, stream) : launch<64, 1, 1, 4, false>(a, stream);
    }
    if (v.key_split == 2) return pad ? launch<128, 1, 2, 4, true>(a, stream) : launch<128, 1, 2, 4, false>(a, stream);
    if (waves == 8) return pad ? launch<128, 1, 1, 8, true>(a, stream) : launch<128, 1, 1, 8, false>(a, stream);
    return pad ? launch<128, 1, 1, 4, true>(a, stream) : launch<128, 1, 1, 4, false>(a, stream);
}
