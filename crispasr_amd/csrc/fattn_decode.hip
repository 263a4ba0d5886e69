// Split-KV MFMA decode kernel for gfx950: few query rows per KV head (beams and/or a GQA group),
// long KV cache, HBM-bound.
//
// A workgroup of 4 waves owns one (KV head, batch, KV split, chunk of 16 query rows); the query rows
// that read this KV head - all queries of all q heads in its GQA group, 16 of them per chunk - are
// the 16 columns of v_mfma_f32_16x16x32_f16 tiles, so K and V are fetched once per KV head and chunk,
// not once per query row (decode steps have one chunk; a short prompt has a few, and each streams the
// head's K/V again).  Each wave walks its share of the split in steps of 32 keys:
//
//   S^T[key, row] = K[key, :] . Q[row, :]^T      A = K from global memory in operand layout
//                                                 (128-bit loads: 16 rows x 64 contiguous bytes)
//   O^T[d,   row] = V[:, d]^T . P^T[:, row]      A = V^T via a wave-private LDS stage written with
//                                                 coalesced 128-bit rows and read back with
//                                                 ds_read_b64_tr_b16; B = P straight from the
//                                                 accumulator registers of the first product
//
// Q8_0 caches are dequantised in registers: the 8 int8 of a lane's chunk are fetched with three
// aligned dword loads and a byte funnel shift (blocks are 34 bytes, so chunks sit at 2 mod 4),
// widened to exact f16 integers with v_perm_b32 + one packed add, and scaled by the block's f16 d
// with one packed multiply (one rounding, = f16(q*d)).  When the rows of a Q8_0 cache are contiguous the
// K bytes of a step are fetched as one coalesced stream of 8- (or 4-)byte units into a wave-private raw
// stage in LDS and the chunks are cut out of LDS instead - three times fewer global load instructions.
// V then skips the f16 stage: it arrives as the same kind of stream, its quants are stored to LDS as bytes - every
// 2-byte piece of a unit written to its place, [key][column] for quants and [block][key] for scales - and read back
// through ds_read_b64_tr_b8, which hands every lane eight consecutive keys of one column - the A operand of the second
// product - to be widened and multiplied by those keys' scales in registers: same values, half the LDS bytes, one
// register stage instead of two.  Q4_0 / Q4_1 / Q5_0 / Q5_1 rows are streamed the same way into raw K and V stages and
// dequantised out of LDS (V into the f16 stage).  Streams and f16 rows are loaded non-temporal: they are read once.
// Loads of the next step are in flight while the current one is consumed.  Waves are merged through LDS, splits by the last
// workgroup of a set where the call has counters for it (fattn_last_of_set), by fattn_merge_kernel otherwise.
//
// Masked calls walk the steps between the first and the last that one of their rows sees, and a step's mask values are
// requested with its K and V: one step for 64 sequences of 500 to 4096 Q8_0 entries (32 query, 8 KV heads of 128) 115 -> 81 us,
// 71 with the sequences paired by length on the CUs (sequence_of_turn), 4.5 TB/s over the entries seen; the bound is what a CU's port
// brings.  (Calls inside a graph.  By box and inputs 65 to 71 us, 4.5 to 4.9 TB/s.)
#include "fattn_row.h"
#include "decode_short.h"

#include <stdlib.h>
#include <type_traits>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float    float4v __attribute__((ext_vector_type(4)));
typedef short    short4v __attribute__((ext_vector_type(4)));

constexpr int   DEC_WAVES   = 4;
constexpr int   DEC_THREADS = DEC_WAVES * 64;
constexpr int   STEP        = 32;                  // keys per wave step
constexpr float LOG2E       = 1.4426950408889634f;
constexpr float SUM_LIMIT   = 4096.0f;             // 8 probabilities per lane and step

// K and V are read once per launch and loaded with stream_load where a wave instruction takes whole lines once - the
// coalesced row streams and f16 rows (64 sequences x 4096 f16 entries: 169 against 188 us).  Per-lane pieces of block
// rows come back to a line several times: the 8-byte pieces and halfword scales of the int8 V stage lose 3-5% when
// marked, and the strided-row forms stay plain with them.
typedef uint32_t u32x2    __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4    __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

// ---- Q8_0 in registers ------------------------------------------------------------------

// the 8 quants of chunk c (0..3) of block blk of a row whose address is a multiple of 4
__device__ __forceinline__ uint2 q8_load_chunk(const char * row, int blk, int c) {
    const int o  = blk * FATTN_Q8_0_BYTES + 2 + c * 8;
    const int sh = o & 3;                                   // 0 or 2
    const uint32_t * p = (const uint32_t *)(row + (o - sh));
    const uint32_t u0 = p[0];
    const uint32_t u1 = p[1];
    const uint32_t u2 = sh ? p[2] : 0u;                     // never read past the row when aligned
    uint2 r;
    r.x = __builtin_amdgcn_alignbyte(u1, u0, sh);
    r.y = __builtin_amdgcn_alignbyte(u2, u1, sh);
    return r;
}

// the same from a raw copy of the rows in LDS (row_off = byte offset of the row inside the stage)
// (row_off is a multiple of 4, so odd blocks start on a dword; UNIFORM_BLK says blk is the same in every lane)
template <bool UNIFORM_BLK>
__device__ __forceinline__ uint4 q8_lds_chunk(const char * stage, int row_off, int blk, int c) {
    const int o  = row_off + blk * FATTN_Q8_0_BYTES + 2 + c * 8;
    const int sh = (blk & 1) ? 0 : 2;
    const uint32_t * p = (const uint32_t *)(stage + (o - sh));
    const uint32_t u0 = p[0], u1 = p[1], u2 = p[2];         // the stage is padded: p[2] is always inside it
    uint4 r;
    if (UNIFORM_BLK && (blk & 1)) {
        r.x = u0;
        r.y = u1;
    } else {
        r.x = __builtin_amdgcn_alignbyte(u1, u0, sh);
        r.y = __builtin_amdgcn_alignbyte(u2, u1, sh);
    }
    r.z = *(const uint16_t *)(stage + row_off + blk * FATTN_Q8_0_BYTES);
    r.w = 0;
    return r;
}

// 4 int8 packed in a dword -> 4 exact f16 integers: bytes become the low mantissa bits of
// 1024 + (q + 128), then 1152 is subtracted
__device__ __forceinline__ void q8_widen(uint32_t w, half2v & lo, half2v & hi) {
    const uint32_t x = w ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(x, 0x64646464u, 0x00050004u);   // {0x64, b1, 0x64, b0}
    const uint32_t b = __builtin_amdgcn_perm(x, 0x64646464u, 0x00070006u);   // {0x64, b3, 0x64, b2}
    const half2v off = {(_Float16)1152.0f, (_Float16)1152.0f};
    lo = __builtin_bit_cast(half2v, a) - off;
    hi = __builtin_bit_cast(half2v, b) - off;
}

__device__ __forceinline__ half8 q8_dequant(uint2 q, uint16_t dbits) {
    const _Float16 d  = __builtin_bit_cast(_Float16, dbits);
    const half2v   d2 = {d, d};
    half2v h0, h1, h2, h3;
    q8_widen(q.x, h0, h1);
    q8_widen(q.y, h2, h3);
    h0 *= d2; h1 *= d2; h2 *= d2; h3 *= d2;
    half8 r;
    r[0] = h0[0]; r[1] = h0[1]; r[2] = h1[0]; r[3] = h1[1];
    r[4] = h2[0]; r[5] = h2[1]; r[6] = h3[0]; r[7] = h3[1];
    return r;
}

// 8 quants of 8 different keys (one column of V) times those keys' scales
__device__ __forceinline__ half8 q8_dequant_keys(uint32_t q0, uint32_t q1, half8 d) {
    half2v h0, h1, h2, h3;
    q8_widen(q0, h0, h1);
    q8_widen(q1, h2, h3);
    half8 r;
    r[0] = h0[0]; r[1] = h0[1]; r[2] = h1[0]; r[3] = h1[1];
    r[4] = h2[0]; r[5] = h2[1]; r[6] = h3[0]; r[7] = h3[1];
    return r * d;
}

// a unit of a streamed row (aux 2: non-temporal, as stream_load)
template <typename T>
__device__ __forceinline__ T buffer_stream(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (sizeof(T) == 16)     return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 2));
    else if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 2));
    else                               return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 2));
}

// raw global data of one 8-element chunk
struct Chunk {
    uint4 v;         // f16: the 8 halves; q8_0: x,y = quants, z = scale bits
};

// Q4_0 / Q4_1 / Q5_0 / Q5_1: x, y = the 8 bytes that hold the chunk's nibbles, shifted so that they sit in the low halves;
// z = d (low) and m (high halfword); w = the chunk's 8 fifth bits.  q0, q1: the 8 bytes at QS + 8 (c % 2) of the block,
// dm: d in the low halfword (and m in the high one), qh: the block's 32 fifth bits, c: which 8 of the block's 32 elements.
__device__ __forceinline__ Chunk narrow_fields(uint32_t q0, uint32_t q1, uint32_t dm, uint32_t qh, int c) {
    Chunk r;
    const int sh = (c & 2) ? 4 : 0;
    r.v.x = (q0 >> sh) & 0x0F0F0F0Fu;
    r.v.y = (q1 >> sh) & 0x0F0F0F0Fu;
    r.v.z = dm;
    r.v.w = (qh >> (c * 8)) & 0xFFu;
    return r;
}

// the same from the block's first 8 bytes h0, h1
template <int TYPE>
__device__ __forceinline__ Chunk narrow_chunk(uint32_t q0, uint32_t q1, uint32_t h0, uint32_t h1, int c) {
    typedef BlockFormat<TYPE> F;
    const uint32_t qh = !F::QH ? 0u : F::QH == 4 ? h1 : __builtin_amdgcn_alignbyte(h1, h0, 2);
    return narrow_fields(q0, q1, F::HAS_M ? h0 : h0 & 0xFFFFu, qh, c);
}

// the same chunk cut out of a raw copy of the rows in LDS (row_off: byte offset of the row inside the stage, a multiple
// of 4; blocks and their quants start on even bytes) with aligned dword reads.  Whether a block starts on a dword or two
// bytes past one depends on the block's index alone - 18- and 22-byte blocks alternate, 20- and 24-byte ones always start
// on one - so with blk a constant after unrolling, every shift here is decided at compile time.  The stage is padded:
// the dword after a pair is always inside it.
template <int TYPE>
__device__ __forceinline__ Chunk narrow_lds_chunk(const char * stage, int row_off, int blk, int c) {
    typedef BlockFormat<TYPE> F;
    const int mis  = (blk * F::BYTES) & 2;                   // bytes from the dword below to the block
    const int misq = (mis + F::QS) & 2;                      // ... to its quants
    const uint32_t * ph = (const uint32_t *)(stage + row_off + blk * F::BYTES - mis);
    const uint32_t * pq = (const uint32_t *)(stage + row_off + blk * F::BYTES + F::QS + (c & 1) * 8 - misq);
    const uint32_t a0 = ph[0];
    uint32_t q0 = pq[0], q1 = pq[1];
    if (misq) {
        const uint32_t q2 = pq[2];
        q0 = __builtin_amdgcn_alignbyte(q1, q0, 2);
        q1 = __builtin_amdgcn_alignbyte(q2, q1, 2);
    }
    const uint32_t dm = F::HAS_M ? a0 : mis ? a0 >> 16 : a0 & 0xFFFFu;
    uint32_t qh = 0;
    if (F::QH == 4) qh = ph[1];                                                    // fifth bits at byte 4
    if (F::QH == 2) qh = mis ? ph[1] : __builtin_amdgcn_alignbyte(ph[1], a0, 2);   // at byte 2
    return narrow_fields(q0, q1, dm, qh, c);
}

// bytes per block of the types the raw stream carries (Q8_0 for the others: they never instantiate it)
template <int TYPE> constexpr int raw_block_bytes() {
    if constexpr (FATTN_IS_BLOCK_TYPE(TYPE)) return BlockFormat<TYPE>::BYTES;
    else return FATTN_Q8_0_BYTES;
}

template <int TYPE>
__device__ __forceinline__ Chunk load_chunk(const char * row, int c) {
    Chunk r;
    if constexpr (TYPE == MI355X_TYPE_F16) {
        r.v = __builtin_bit_cast(uint4, stream_load<u32x4>(row + c * 16));
    } else if constexpr (TYPE == MI355X_TYPE_Q8_0) {
        const uint2 q = q8_load_chunk(row, c >> 2, c & 3);
        r.v.x = q.x;
        r.v.y = q.y;
        r.v.z = *(const uint16_t *)(row + (c >> 2) * FATTN_Q8_0_BYTES);
        r.v.w = 0;
    } else {
        typedef BlockFormat<TYPE> F;
        const char * blk = row + (c >> 2) * F::BYTES;
        const int    j0  = (c & 3) * 8;                                   // first element of the chunk inside its block
        const u32x2_a2 q = *(const u32x2_a2 *)(blk + F::QS + (j0 & 8));     // elements j and j + 16 share a byte
        const u32x2_a2 h = *(const u32x2_a2 *)blk;                          // the block's first 8 bytes: d [, m] [, fifth bits]
        r = narrow_chunk<TYPE>(q[0], q[1], h[0], h[1], c & 3);
    }
    return r;
}

// 4 unsigned bytes -> 4 exact f16 integers minus `off`: a byte becomes the low mantissa bits of 1024 + b
__device__ __forceinline__ void u8_widen(uint32_t w, float off, half2v & lo, half2v & hi) {
    const uint32_t a = __builtin_amdgcn_perm(w, 0x64646464u, 0x00050004u);   // {0x64, b1, 0x64, b0}
    const uint32_t b = __builtin_amdgcn_perm(w, 0x64646464u, 0x00070006u);   // {0x64, b3, 0x64, b2}
    const _Float16 o = (_Float16)(1024.0f + off);
    const half2v   o2 = {o, o};
    lo = __builtin_bit_cast(half2v, a) - o2;
    hi = __builtin_bit_cast(half2v, b) - o2;
}

template <int TYPE>
__device__ __forceinline__ half8 chunk_to_half8(const Chunk & r) {
    if constexpr (TYPE == MI355X_TYPE_F16) {
        return __builtin_bit_cast(half8, r.v);
    } else if constexpr (TYPE == MI355X_TYPE_Q8_0) {
        return q8_dequant(make_uint2(r.v.x, r.v.y), (uint16_t)r.v.z);
    } else {
        typedef BlockFormat<TYPE> F;
        uint32_t x = r.v.x, y = r.v.y;
        if (F::QH) {       // bit i of the byte of fifth bits -> bit 4 of byte i
            x |= (((r.v.w & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
            y |= (((r.v.w >> 4) * 0x00204081u) & 0x01010101u) << 4;
        }
        half2v h0, h1, h2, h3;
        const float off = F::HAS_M ? 0.0f : (float)(F::LEVELS / 2);
        u8_widen(x, off, h0, h1);
        u8_widen(y, off, h2, h3);
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)(r.v.z & 0xFFFFu));
        const half2v   d2 = {d, d};
        if (F::HAS_M) {    // f16(q * d + m), one rounding
            const _Float16 m = __builtin_bit_cast(_Float16, (uint16_t)(r.v.z >> 16));
            const half2v   m2 = {m, m};
            h0 = __builtin_elementwise_fma(h0, d2, m2); h1 = __builtin_elementwise_fma(h1, d2, m2);
            h2 = __builtin_elementwise_fma(h2, d2, m2); h3 = __builtin_elementwise_fma(h3, d2, m2);
        } else {
            h0 *= d2; h1 *= d2; h2 *= d2; h3 *= d2;
        }
        half8 o;
        o[0] = h0[0]; o[1] = h0[1]; o[2] = h1[0]; o[3] = h1[1];
        o[4] = h2[0]; o[5] = h2[1]; o[6] = h3[0]; o[7] = h3[1];
        return o;
    }
}

// row pitch in bytes of the int8 V stage: the 16 rows one half of a transpose read touches start 4 banks apart
template <int D> constexpr int v8_pitch() { return D == 128 ? 136 : 80; }

// Waves a SIMD is to hold, at least and at most, where the compiler's own guess is a bad one.  Streamed 64-wide rows come to
// a register or two above or below 128, with which four workgroups share a CU, for three (Q4_0, 64 sequences x 16 heads
// against 160 masked entries: 10.7 us with 129 registers, 8.5 with 128; Q5_0 takes 143 under a mask and would spill).  The LDS
// of streamed 128-wide rows of narrow types holds two workgroups: a schedule that keeps registers free for a third is slower
// for nothing (Q4_0, 64 sequences of 500 to 4096 entries, 167 registers 73.4 us, 177 registers 67.1).
template <int D, int TYPE, bool RAW> constexpr int decode_waves_min() {
    return D == 64 && RAW && (TYPE == MI355X_TYPE_Q4_0 || TYPE == MI355X_TYPE_Q4_1 || TYPE == MI355X_TYPE_Q5_1) ? 4 : 2;
}
template <int D, bool RAW, bool V8> constexpr int decode_waves_max() { return D == 128 && RAW && !V8 ? 2 : 8; }

// LDS bytes per workgroup: the per-wave f16 V stages, plus per-wave raw K and V stages when RAW; with V8 the V side is
// one int8 stage and the scales of its 32 x D/32 blocks instead
template <int D, int TYPE, bool RAW, bool V8>
constexpr int decode_lds_bytes() {
    constexpr int RS     = D / 32 * raw_block_bytes<TYPE>();
    constexpr int RAWSZ  = (STEP * RS + 511) / 512 * 512 + 64;                      // 9 x 64 units, padded
    constexpr int wave   = V8 ? RAWSZ + STEP * v8_pitch<D>() + D / 32 * STEP * 2
                              : STEP * (D + 32) * 2 + (RAW ? 2 * RAWSZ : 0);
    constexpr int stage  = DEC_WAVES * wave;
    constexpr int red    = DEC_WAVES * 16 * (D + 4 + 2) * 4;
    return stage > red ? stage : red;
}

// Where the 2-byte pieces of a step's 32 Q8_0 rows go in the int8 V stage, as offsets from the wave's LDS block: byte o
// of the step is byte o % RS of row o / RS; byte 0 of a 34-byte block is its scale's (-> f16 [block][key] behind the
// stage), bytes 2.. are its quants' (-> [key][column]).  Indexed by piece o / 2, padded to whole 64-lane loads of units.
template <int D>
struct V8Places {
    static constexpr int RS = D / 32 * FATTN_Q8_0_BYTES, UNIT = RS % 8 == 0 ? 8 : 4;
    static constexpr int UNITS = (STEP * RS / UNIT + 63) / 64 * 64;
    static constexpr int RAWSZ = (STEP * RS + 511) / 512 * 512 + 64;
    uint16_t at[UNITS * UNIT / 2];
};
template <int D>
constexpr V8Places<D> v8_places() {
    typedef V8Places<D> P;
    P t{};
    for (int o = 0; o < STEP * P::RS; o += 2) {
        const int row = o / P::RS, rem = o % P::RS, blk = rem / FATTN_Q8_0_BYTES, ib = rem % FATTN_Q8_0_BYTES;
        t.at[o / 2] = (uint16_t)(ib == 0 ? P::RAWSZ + STEP * v8_pitch<D>() + (blk * STEP + row) * 2
                                         : P::RAWSZ + row * v8_pitch<D>() + blk * 32 + ib - 2);
    }
    return t;
}
template <int D> __device__ const V8Places<D> v8_places_table = v8_places<D>();

// The sequence whose turn it is where they go by length (decode_turns; at most 128).  Lengths are counted in eighths: eight keys of
// every sequence's mask, two a wave, in the last query's row (what a count is off by, or a mask that does not end a sequence, costs
// balance and nothing else: every workgroup counts the same, and the places are a permutation).  A look costs 1.3 us where nothing else
// runs on the CU, so the first round takes the sequences in their own order, and the next ones, whose look hides behind it, make up for that.
__device__ __forceinline__ int sequence_of_turn(const FattnArgs & a, int turn, int first, char * lds) {
    if (turn < first) return turn;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int * counts = (int *)lds;                     // [wave][128]
    const bool more = a.B > 64;
#pragma unroll
    for (int g = 0; g < 2; g++)
        if (g == 0 || more) {
            const int        b   = min(g * 64 + lane, a.B - 1);
            const uint16_t * row = (const uint16_t *)(a.mask + (int64_t)b * a.nbm3 + (int64_t)(a.Nq - 1) * a.nbm1);
            const uint16_t v0 = row[(int)((int64_t)(wave * 4 + 1) * a.Nkv >> 4)], v1 = row[(int)((int64_t)(wave * 4 + 3) * a.Nkv >> 4)];
            counts[wave * 128 + g * 64 + lane] = (v0 != 0xFC00u) + (v1 != 0xFC00u);
        }
    __syncthreads();
    int seen[2] = {0, -1};
#pragma unroll
    for (int w = 0; w < DEC_WAVES; w++) seen[0] += counts[w * 128 + lane];
    if (lane >= a.B) seen[0] = -1;
    if (more && 64 + lane < a.B) {
        seen[1] = 0;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; w++) seen[1] += counts[w * 128 + 64 + lane];
    }
    __syncthreads();                               // the stages of the key loop lie where the counts do

    // places by length, the longest first, among the sequences [from, to): of sequence `lane` and of 64 + lane
    int place[2];
    auto rank = [&](int from, int to) __attribute__((always_inline)) {
        place[0] = place[1] = -1;
        int n = 0;
#pragma unroll
        for (int eighths = 8; eighths >= 0; eighths--)
#pragma unroll
            for (int g = 0; g < 2; g++)
                if (g == 0 || more) {
                    const bool     one   = seen[g] == eighths && g * 64 + lane >= from && g * 64 + lane < to;
                    const uint64_t those = __ballot(one);
                    const int      at    = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(those >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)those, 0));
                    if (one) place[g] = at;
                    n += __popcll(those);
                }
    };
    const int behind = turn - first, pairs = min(first, a.B - first);      // (pairs <= 64)
    int want = behind;
    if (behind < pairs) {                          // beside sequence `behind`: the longest of those gets the shortest of these
        rank(0, pairs);
        want = pairs - 1 - __builtin_amdgcn_readlane(place[0], behind);
    }
    rank(first, a.B);
    const uint64_t low = __ballot(place[0] == want), high = __ballot(place[1] == want);
    return low ? __builtin_ctzll(low) : high ? 64 + __builtin_ctzll(high) : 0;
}

// V8 (with RAW): V's quants go to LDS as bytes and come back through ds_read_b64_tr_b8 already in operand layout
// (8 consecutive keys of one column per lane).  The transposing read ignores the low three address bits and the quants
// of block b start at byte 34 b + 2 of a row, so the rows cannot stay as they are in memory: V arrives as the same
// coalesced stream as K, and each 2-byte piece of a unit is written to its place - a pair of quants to [key][column],
// a scale to [block][key] - by one ds_write_b16 whose address depends on the lane alone (read from a table behind the
// first K/V request: computing the 36 of them costs more instructions than a 32-key step).
// PAD: f16 rows of a.Dv elements (a multiple of 8 below D) read in place: the chunks of a row behind Dv are zeros in the
// registers, q is read and dst written up to Dv.  An instantiation of its own: the others stay the code they were.
// SHORT: the arguments came as DecodeShort, the grid is (split, KV head, batch), and there is one chunk of rows; `first`: decode_turns.
// DEEP (f16 rows, SHORT, no mask): the rows of two steps are under way while a third is worked on; q is asked for first.
template <int D, int TYPE, bool MASK, bool RAW, bool V8, bool PAD, bool SHORT, bool DEEP = false>
__device__ __forceinline__ void decode_body(const FattnArgs & a, int first) {
    static_assert(!PAD || (TYPE == MI355X_TYPE_F16 && !RAW && !V8), "other head sizes: f16 rows, read per lane");
    static_assert(!V8 || RAW, "the int8 V stage belongs to the streamed Q8_0 path");
    static_assert(!DEEP || (SHORT && !MASK && TYPE == MI355X_TYPE_F16), "see above");
    constexpr int KS  = D / 32;                    // reduction steps of Q.K^T (one Q8_0 block each)
    constexpr int DBK = D / 16;                    // 16-wide blocks of the output's d
    constexpr int CH  = D / 8;                     // chunks per row
    constexpr int NV  = STEP * CH / 64;            // V chunks per lane and step
    constexpr int PV  = D + 32;                    // LDS pitch in halves: 64 mod 128 bytes
    // raw streaming of contiguous rows of blocks: UNIT-byte loads, NU per lane and tensor and step
    constexpr int BB    = raw_block_bytes<TYPE>();
    constexpr int RS    = D / 32 * BB;
    constexpr int UNIT  = RS % 8 == 0 ? 8 : 4;
    constexpr int UPS   = STEP * RS / UNIT;        // units per full step
    constexpr int NU    = (UPS + 63) / 64;
    constexpr int RAWSZ = (STEP * RS + 511) / 512 * 512 + 64;
    static_assert(!RAW || FATTN_IS_BLOCK_TYPE(TYPE), "raw streaming is for rows of blocks");
    static_assert(!V8 || TYPE == MI355X_TYPE_Q8_0, "the int8 V stage holds Q8_0 quants");
    static_assert(NU * 64 * UNIT <= RAWSZ, "raw stage too small");

    // the per-wave stages; after the key loop the same memory carries the cross-wave reduction
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int VP8 = v8_pitch<D>();
    constexpr int PCS = UNIT / 2;                  // (V8) 2-byte pieces per unit
    // unmasked: the request of Q ahead of the first K/V request.  (Not for 64-wide Q8_0, whose waves are bound by their steps: 3 rows x 16 heads x
    // 16 sequences against 500 entries 6.70 us with Q behind it, 6.97 ahead, 32 query and 8 KV heads x 16 against 4000 15.4, 16.1.)
    constexpr bool Q_FIRST = RAW && !(V8 && D == 64);
    constexpr bool ONE = V8;                       // one register stage: the next step is requested once this one is in LDS
                                                   // (two stages, as the other forms have: 102-104 against 99 us at 64 x 4096)
    constexpr int WAVE_BYTES = V8 ? RAWSZ + STEP * VP8 + KS * STEP * 2 : STEP * PV * 2 + (RAW ? 2 * RAWSZ : 0);
    char * const wave_mem = smem + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * WAVE_BYTES;
    _Float16 * v_stage = (_Float16 *)wave_mem;                          // (!V8)
    char * k_rawst     = V8 ? wave_mem : wave_mem + STEP * PV * 2;
    char * v_rawst     = k_rawst + RAWSZ;                               // (!V8)
    char * v8_stage    = wave_mem + RAWSZ;                              // (V8) [32 keys][VP8]
    char * vsc_stage   = v8_stage + STEP * VP8;                         // (V8) f16 [KS][32 keys]
    // (rows D + 4 floats apart: the 16 columns of a 128-bit store start 4 banks apart)
    float (*red_o)[16][D + 4]      = (float (*)[16][D + 4])smem;
    float (*red_ml)[16][2]         = (float (*)[16][2])(smem + DEC_WAVES * 16 * (D + 4) * 4);

    const int tid  = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);     // uniform: loop control and row bases stay scalar
    const int lane = tid & 63;
    const int j    = lane & 15;                    // query column
    const int g4   = lane >> 4;

    // workgroup = (split, 16-row chunk, KV head, batch), splits fastest.  With more than one chunk of rows per KV head the
    // chunks of one (split, KV head, batch) read the same keys: workgroups go to the 8 XCDs round-robin, each with its own
    // L2, so those chunks are numbered to follow each other on ONE XCD (the grid is rounded up to whole rounds of 8;
    // the spare workgroups leave here, before any barrier, and belong to no set of the merge).
    int     split, chunk, hk, b;
    int64_t set;                                   // index of (chunk, KV head, batch): the merge's counter
    // (divisions by multiply and shift: a call that is one or two steps long spends 0.3 us on five ordinary ones)
    chunk = 0;
    if constexpr (SHORT) {
        split = (int)blockIdx.x;
        hk    = (int)blockIdx.y;
        b     = MASK && first ? sequence_of_turn(a, (int)blockIdx.z, first, smem) : (int)blockIdx.z;
        set   = (int64_t)b * a.Hkv + hk;
    } else {
        uint32_t pair = blockIdx.x;
        if (a.q_chunks != 1) {
            const uint32_t w  = blockIdx.x >> 3;
            const uint32_t wc = divide(w, a.by_chunks);
            pair  = wc * 8u + (blockIdx.x & 7u);
            chunk = (int)(w - wc * (uint32_t)a.q_chunks);
            if (pair >= (uint32_t)a.n_splits * (uint32_t)a.Hkv * (uint32_t)a.B) return;      // (<= the grid)
        }
        const uint32_t head = divide(pair, a.by_splits);
        b     = (int)divide(head, a.by_hkv);
        split = (int)(pair - head * (uint32_t)a.n_splits);
        hk    = (int)head - b * a.Hkv;
        set   = (int64_t)head * a.q_chunks + chunk;
    }
    const int bk = SHORT ? b : (int)divide((uint32_t)b, a.by_bq);
    // row / gqa (SHORT: both at most 16, and (row + 1/2) / gqa is never near a whole number)
    const float per_row = SHORT ? __builtin_amdgcn_rcpf((float)a.gqa) : 0.0f;
    auto query_of = [&](int row) __attribute__((always_inline)) {
        return SHORT ? (int)(((float)row + 0.5f) * per_row) : (int)divide((uint32_t)row, a.by_gqa);
    };

    // row r = iq1 * gqa + gg of this KV head  <->  query iq1 of q head hk*gqa + gg; column j is row chunk*16 + j
    const int  R      = a.Nq * a.gqa;
    const int  row0   = chunk * 16;
    const bool col_ok = row0 + j < R;
    const int  jc     = col_ok ? row0 + j : row0;
    const int  iq1    = query_of(jc);
    const int  h      = hk * a.gqa + jc - iq1 * a.gqa;

    const int k_begin = split * a.keys_per_split;
    const int k_end   = min(a.Nkv, k_begin + a.keys_per_split);

    half8 qreg[KS];
    const char * kbase = a.k + (int64_t)hk * a.nbk2 + (int64_t)bk * a.nbk3;
    const char * vbase = a.v + (int64_t)hk * a.nbv2 + (int64_t)bk * a.nbv3;
    const char * mhead = MASK ? a.mask + (int64_t)(SHORT ? h : h - (int)divide((uint32_t)h, a.by_hm) * a.Hm) * a.nbm2 +
                                (int64_t)(SHORT ? b : b - (int)divide((uint32_t)b, a.by_bm) * a.Bm) * a.nbm3
                              : nullptr;
    const uint16_t * mrow = (const uint16_t *)(mhead + (int64_t)iq1 * a.nbm1);
    const float mslope = MASK ? fattn_slope(a, h) * LOG2E : 0.0f;

    float4v oacc[DBK];
#pragma unroll
    for (int db = 0; db < DBK; db++) oacc[db] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    float m = 0.0f, l = 0.0f;
    bool  have = false;

    const int n_steps = k_end > k_begin ? (k_end - k_begin + STEP - 1) / STEP : 0;

    // (MASK) Which of the wave's steps any of the chunk's rows sees: a step without a visible key adds exact zeros, so the wave
    // walks those between its first and its last visible one.  Two requests of 8 keys a lane, four lanes a step, see one row
    // over 32 steps of the wave (a split of 4096 keys) or 8 rows of a mask without heads over 4 (512 keys).  Other splits count
    // every step as visible, and so does a slope that has underflowed to zero (0 * -inf is NaN, as it is on the CPU).  Reads stay
    // inside [k_begin, k_end) by moving the last ones back: at worst a step is taken for visible because the one before it is.
    // A look costs 0.3 us and is worth it from two steps a wave on, where it can save one: 5 beams against 140 entries, 20 heads
    // of 64, 4.8 us without it, 5.2 with it, 6.1 where every wave looked at all of its split; a 2048-entry cache of which 100
    // are written, 16 query, 8 KV heads of 128, 10.3, 9.2 and 9.9 us.  Splits of one step a wave never look.
    const uint32_t EXCLUDED2 = 0xFC00FC00u;                 // two masked-out keys
    int        walk = wave, walk_end = n_steps;             // the steps that the wave walks
    const int  iq_0    = MASK ? query_of(row0) : 0;
    const int  iq_1    = MASK ? query_of(min(row0 + 15, R - 1)) : 0;
    const bool one_row = iq_1 == iq_0;
    const bool looking = MASK && n_steps > DEC_WAVES && (one_row ? n_steps <= 128 : n_steps <= 16 && iq_1 - iq_0 < 8) && (a.Hm == 1 || R == 1) &&
                         __builtin_amdgcn_ballot_w64(!(mslope > 0.0f)) == 0;
    auto look_key = [&](int i) __attribute__((always_inline)) {         // the first of the lane's 8 keys of request i
        const int t = one_row ? i * 16 + (lane >> 2) : (lane >> 2) & 3;
        return k_begin + (wave + t * DEC_WAVES) * STEP + (lane & 3) * 8;
    };
    auto look_at = [&](int i) __attribute__((always_inline)) {
        const int row = one_row ? iq_0 : min(iq_0 + i * 4 + (lane >> 4), iq_1);
        return *(const u32x4_a2 *)(mhead + (int64_t)row * a.nbm1 + (int64_t)min(look_key(i), k_end - 8) * 2);
    };

    // loads of one step: K in operand layout (key = kb*16 + j, chunk = ks*4 + g4), V in row order
    Chunk kraw[2][RAW ? 1 : 2][RAW ? 1 : KS];
    Chunk vraw[2][RAW ? 1 : NV];
    typedef typename std::conditional<UNIT == 8, u32x2, uint32_t>::type unit_t;
    // (V8 keeps one register stage: index 0 whatever the step's stage number)
    unit_t kun[2][RAW ? NU : 1], vun[2][RAW ? NU : 1];
    // (V8) LDS offsets from wave_mem of the pieces of this lane's V units, two to a register
    uint32_t vdst[V8 ? NU : 1][V8 ? PCS / 2 : 1];
    // mask values of the lane's eight keys of the step, in the order of its scores
    u32x2_a2 mraw[2][MASK ? 2 : 1];
    // (DEEP) Rows through a buffer that ends with the step's last valid one, or holds nothing behind the wave's last step: the request
    // needs no branch.  With one, the compiler cannot count what is on its way behind a stage and waits for everything at each step, so
    // that no step's rows were under way during another.  A lane's offsets of K's rows j and V's, the same for every step:
    const uint32_t nb1  = DEEP ? (uint32_t)a.nbk1 : 0;          // (K's and V's, below 64 MiB)
    const uint32_t koff = (uint32_t)j * nb1 + g4 * 16, voff = (uint32_t)(lane / CH) * nb1 + lane % CH * 16;
    // a partial last step: its loads are clamped to the last valid row (branch-free, in bounds) or give zeros behind it, and
    // the keys they stand for are excluded in the step
    auto issue = [&](int it, auto stage) __attribute__((always_inline)) {
        constexpr int s = decltype(stage)::value;
        const bool on = !DEEP || it < walk_end;
        const int  j0 = k_begin + (on ? it : 0) * STEP;
        // (One branch for the eight values where a step's registers are many; the int8 V form, with one register stage, is up to
        //  3% faster on large batches with one branch for each four.)
        if constexpr (MASK && V8) {
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const int key = j0 + g4 * 8 + kb * 4;
                if (j0 + STEP <= k_end) {
                    mraw[0][kb] = *(const u32x2_a2 *)(mrow + key);
                } else {
#pragma unroll
                    for (int r = 0; r < 2; r++)
                        mraw[0][kb][r] = (uint32_t)mrow[min(key + 2 * r, k_end - 1)] | (uint32_t)mrow[min(key + 2 * r + 1, k_end - 1)] << 16;
                }
            }
        } else if constexpr (MASK) {
            if (__builtin_expect(j0 + STEP <= k_end, 1)) {
#pragma unroll
                for (int kb = 0; kb < 2; kb++) mraw[s][kb] = *(const u32x2_a2 *)(mrow + j0 + kb * 16 + g4 * 4);
            } else {
                uint32_t w[8];
#pragma unroll
                for (int e = 0; e < 8; e++) w[e] = mrow[min(j0 + (e >> 2) * 16 + g4 * 4 + (e & 3), k_end - 1)];
#pragma unroll
                for (int e = 0; e < 8; e += 2) mraw[s][e >> 2][(e >> 1) & 1] = w[e] | w[e + 1] << 16;
            }
        }
        if (RAW) {
            // One coalesced stream per tensor, through a buffer that ends with the step's last valid row: what lies behind it are
            // zeros, scales and minima among them, and the 2 * NU loads share one offset (its lane number through an asm, or
            // each of the loop's would have its own).
            const uint32_t bytes = (uint32_t)min(STEP, k_end - j0) * RS;
            const auto     kb = fattn_buffer(kbase + (int64_t)j0 * RS, bytes), vb = fattn_buffer(vbase + (int64_t)j0 * RS, bytes);
            uint32_t ln = (uint32_t)lane;
            asm volatile("" : "+v"(ln));
#pragma unroll
            for (int i = 0; i < NU; i++) {
                kun[ONE ? 0 : s][i] = buffer_stream<unit_t>(kb, (ln + i * 64) * UNIT);
                vun[ONE ? 0 : s][i] = buffer_stream<unit_t>(vb, (ln + i * 64) * UNIT);
            }
            return;
        }
        if constexpr (DEEP) {
            const uint32_t bytes = on ? (uint32_t)(min(STEP, k_end - j0) - 1) * nb1 + (uint32_t)(PAD ? a.Dv : D) * 2 : 0;
            const auto     kbuf = fattn_buffer(kbase + (int64_t)j0 * nb1, bytes), vbuf = fattn_buffer(vbase + (int64_t)j0 * nb1, bytes);
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    kraw[s][kb][ks].v = buffer_stream<uint4>(kbuf, !PAD || (ks * 4 + g4) * 8 < a.Dv ? koff + kb * 16 * nb1 + ks * 64 : FATTN_NO_ADDRESS);
#pragma unroll
            for (int i = 0; i < NV; i++)
                vraw[s][i].v = buffer_stream<uint4>(vbuf, !PAD || lane % CH * 8 < a.Dv ? voff + i * (64 / CH) * nb1 : FATTN_NO_ADDRESS);
            return;
        }
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            const int key = min(j0 + kb * 16 + j, k_end - 1);
            const char * row = kbase + (int64_t)key * a.nbk1;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                if (!PAD || (ks * 4 + g4) * 8 < a.Dv) kraw[s][kb][ks] = load_chunk<TYPE>(row, ks * 4 + g4);
                else                                  kraw[s][kb][ks].v = make_uint4(0u, 0u, 0u, 0u);
            }
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int flat = i * 64 + lane;
            const int key  = min(j0 + flat / CH, k_end - 1);
            if (!PAD || (flat % CH) * 8 < a.Dv) vraw[s][i] = load_chunk<TYPE>(vbase + (int64_t)key * a.nbv1, flat % CH);
            else                                vraw[s][i].v = make_uint4(0u, 0u, 0u, 0u);
        }
    };

    typedef std::integral_constant<int, 0> S0;

    // one step of 32 keys out of register stage s; the wave's following step `nxt` is requested into the other stage
    // (DEEP: the one behind that into this stage, once its rows have gone on; nxt < 0: none)
    auto step = [&](const int it, const int nxt, auto stage) __attribute__((always_inline)) {
        constexpr int s = decltype(stage)::value;
        const int  j0   = k_begin + it * STEP;
        const bool tail = j0 + STEP > k_end;                  // wave-uniform
        // the following step's loads: into the other register stage, or (V8) into this one as soon as it is in LDS
        if (!ONE && !DEEP && nxt < walk_end) issue(nxt, std::integral_constant<int, 1 - s>{});
        u32x2_a2 mcur[2];                                     // (V8's next request overwrites the stage)
        if (MASK) {
            mcur[0] = mraw[ONE ? 0 : s][0];
            mcur[1] = mraw[ONE ? 0 : s][MASK ? 1 : 0];
        }

        if (RAW) {
#pragma unroll
            for (int i = 0; i < NU; i++) {
                *(unit_t *)(k_rawst + (i * 64 + lane) * UNIT) = kun[ONE ? 0 : s][i];
                if (!V8) *(unit_t *)(v_rawst + (i * 64 + lane) * UNIT) = vun[s][i];
            }
            if (V8) {
#pragma unroll
                for (int i = 0; i < NU; i++) {
                    if ((i + 1) * 64 > UPS && i * 64 + lane >= UPS) continue;      // past the step's 32 rows
                    uint32_t w[2];
                    if constexpr (UNIT == 8) { w[0] = vun[ONE ? 0 : s][i][0]; w[1] = vun[ONE ? 0 : s][i][1]; }
                    else                     { w[0] = vun[ONE ? 0 : s][i]; w[1] = 0; }
#pragma unroll
                    for (int k = 0; k < PCS; k++) {
                        const uint32_t dst = k % 2 ? vdst[i][k / 2] >> 16 : vdst[i][k / 2] & 0xFFFFu;
                        *(uint16_t *)(wave_mem + dst) = (uint16_t)(k % 2 ? w[k / 2] >> 16 : w[k / 2]);
                    }
                }
            }
            if (ONE && nxt < walk_end) issue(nxt, stage);
            __builtin_amdgcn_wave_barrier();
        }
        // ---- S^T = K . Q^T ------------------------------------------------------------------
        float4v sc[2];
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            sc[kb] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                Chunk c;
                // (V8: row i of tile kb is key (i / 4) * 8 + kb * 4 + i % 4, so that a lane's eight scores are eight
                //  consecutive keys, the order in which the transposing read hands out V)
                if (RAW && TYPE == MI355X_TYPE_Q8_0) c.v = q8_lds_chunk<true>(k_rawst, (V8 ? (j >> 2) * 8 + kb * 4 + (j & 3) : kb * 16 + j) * RS, ks, g4);
                else if (RAW) c = narrow_lds_chunk<RAW ? TYPE : MI355X_TYPE_Q4_0>(k_rawst, (kb * 16 + j) * RS, ks, g4);
                else     c = kraw[s][kb][ks];
                sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(chunk_to_half8<TYPE>(c), qreg[ks], sc[kb], 0, 0, 0);
            }
        }
        // V rows into this wave's LDS stage (f16, dequantised when the cache is Q8_0)
#pragma unroll
        for (int i = 0; i < (V8 ? 0 : NV); i++) {
            const int flat = i * 64 + lane;
            Chunk c;
            if (RAW && TYPE != MI355X_TYPE_Q8_0) {
                // one block of 16 rows per pass (4 lanes per row), so that the block index is a constant: pass i takes
                // block i % KS of rows 16 (i / KS) ... + 15
                const int row = (i / KS) * 16 + (lane >> 2), ch = (i % KS) * 4 + (lane & 3);
                c = narrow_lds_chunk<RAW ? TYPE : MI355X_TYPE_Q4_0>(v_rawst, row * RS, i % KS, lane & 3);
                *(half8 *)&v_stage[row * PV + ch * 8] = chunk_to_half8<TYPE>(c);
                continue;
            }
            if (RAW) c.v = q8_lds_chunk<false>(v_rawst, (flat / CH) * RS, (flat % CH) >> 2, (flat % CH) & 3);
            else     c = vraw[s][i];
            *(half8 *)&v_stage[(flat / CH) * PV + (flat % CH) * 8] = chunk_to_half8<TYPE>(c);
        }
        if (DEEP && nxt >= 0) issue(nxt, stage);
        __builtin_amdgcn_wave_barrier();      // LDS runs a wave's instructions in order; keep the compiler from reordering

        // lane holds keys j0 + kb*16 + g4*4 + r of column j (V8: j0 + g4*8 + kb*4 + r)
        float sv[8];
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = V8 ? j0 + g4 * 8 + kb * 4 + r : j0 + kb * 16 + g4 * 4 + r;
                float x = sc[kb][r];
                if (MASK) x = fmaf(mslope, h2f_bits((uint16_t)(mcur[kb][r >> 1] >> (16 * (r & 1)))), x);
                if (tail && key >= k_end) x = -INFINITY;
                sv[kb * 4 + r] = x - m;
            }

        // ---- P = 2^(s - m): no maximum unless the step's sum says the reference fell behind -----
        half8 preg;
        float lsum;
        const half2v ones = {(_Float16)1.0f, (_Float16)1.0f};
        auto exp_step = [&]() {
            float acc = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                half2v p2;
                p2[0] = (_Float16)__builtin_amdgcn_exp2f(sv[e]);
                p2[1] = (_Float16)__builtin_amdgcn_exp2f(sv[e + 1]);
                acc = __builtin_amdgcn_fdot2(p2, ones, acc, false);
                preg[e] = p2[0];
                preg[e + 1] = p2[1];
            }
            lsum = acc;
        };
        exp_step();
        const bool redo = !(lsum <= SUM_LIMIT) || !have;
        if (__builtin_amdgcn_ballot_w64(redo) != 0) {
            float mx = sv[0];
#pragma unroll
            for (int e = 1; e < 8; e++) mx = fmaxf(mx, sv[e]);
            mx = fmaxf(mx, xor_shuffle(mx, 16));          // the four lanes of a column must agree
            mx = fmaxf(mx, xor_shuffle(mx, 32));
            float delta = 0.0f;
            if (mx > -INFINITY) {
                delta = have ? fmaxf(mx, 0.0f) : mx;
                have = true;
            }
            const float f = __builtin_amdgcn_exp2f(-fabsf(delta));      // (a first reference far below zero: nothing to scale, and 0 * inf is not 0)
            m += delta;
            l *= f;
#pragma unroll
            for (int db = 0; db < DBK; db++) oacc[db] *= f;
#pragma unroll
            for (int e = 0; e < 8; e++) sv[e] -= delta;
            exp_step();
        }
        l += lsum;

        // ---- O^T += V^T . P^T: transpose reads of the stage, 16 d at a time --------------------------
        if (V8) {
            half8 vsc[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ks++) vsc[ks] = *(const half8 *)(vsc_stage + (ks * STEP + g4 * 8) * 2);
            // lane r of a group of 16 addresses key r / 2, columns 8 (r % 2) ..: the group receives keys g4*8 .. +7 x 16 columns
            const char * p0 = v8_stage + (g4 * 8 + (j >> 1)) * VP8 + (j & 1) * 8;
#pragma unroll
            for (int db = 0; db < DBK; db++) {
                typedef int int2v __attribute__((ext_vector_type(2)));
                const int2v q = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) int2v *)(p0 + db * 16));
                const half8 va = q8_dequant_keys((uint32_t)q[0], (uint32_t)q[1], vsc[db >> 1]);
                oacc[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, preg, oacc[db], 0, 0, 0);
            }
        } else {
            const int kr = g4 * 4 + (j >> 2);
#pragma unroll
            for (int db = 0; db < DBK; db++) {
                const _Float16 * p0 = &v_stage[kr * PV + db * 16 + (j & 3) * 4];
                const _Float16 * p1 = p0 + 16 * PV;
                const half4 lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)p0));
                const half4 hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)p1));
                const half8 va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                oacc[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, preg, oacc[db], 0, 0, 0);
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    // ---- Q: requested here and converted to f16 B operands, in log2 units, once the loads that follow are on their way ------
    float qraw[KS][8];
    auto request_q = [&]() __attribute__((always_inline)) {
        const float * qrow = (const float *)(a.q + (int64_t)iq1 * a.nbq1 + (int64_t)h * a.nbq2 + (int64_t)b * a.nbq3);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            // (PAD: every lane reads 8 elements that exist, its own or the row's first 8 where it has none, and the lanes
            //  without scale them by zero: under a guard each, the 8 * KS loads waited for one another - 2 us per call.  A q row
            //  with inf or NaN in it gives NaN either way.)
            const float * q8 = qrow + (!PAD || ks * 32 + g4 * 8 < a.Dv ? ks * 32 + g4 * 8 : 0);
#pragma unroll
            for (int e = 0; e < 8; e++) qraw[ks][e] = q8[e];
        }
    };
    auto convert_q = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const float qs = !PAD || ks * 32 + g4 * 8 < a.Dv ? a.scale * LOG2E : 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) qreg[ks][e] = (_Float16)(qraw[ks][e] * qs);
        }
    };

    // The look at the mask and Q go out ahead of the first K/V request, that ahead of their answers, so that all of them are
    // one round trip; the request is for the wave's first step, seen or not.
    if constexpr (MASK) {
        u32x4_a2 look[2] = {{EXCLUDED2, EXCLUDED2, EXCLUDED2, EXCLUDED2}, {EXCLUDED2, EXCLUDED2, EXCLUDED2, EXCLUDED2}};
        if (looking) {
            look[0] = look_at(0);
            if (one_row ? n_steps > 64 : iq_1 - iq_0 >= 4) look[1] = look_at(1);
        }
        request_q();
        // (a loop of one turn, or of two where the wave's first step is not seen: the request exists once)
        for (bool asked = false;; asked = true) {
            if (walk < walk_end) issue(walk, S0{});
            if (!looking || asked) break;
            uint64_t seen[2];                               // bits 4 t .. 4 t + 3: keys of the wave's step t (one row)
#pragma unroll
            for (int i = 0; i < 2; i++)
                seen[i] = __builtin_amdgcn_ballot_w64(look_key(i) < k_end && ((look[i][0] ^ EXCLUDED2) | (look[i][1] ^ EXCLUDED2) |
                                                                              (look[i][2] ^ EXCLUDED2) | (look[i][3] ^ EXCLUDED2)) != 0);
            if (!one_row) {                                 // 16 bits a row
                uint64_t v = seen[0] | seen[1];
                v |= v >> 32;
                v |= v >> 16;
                seen[0] = v & 0xFFFFu;
                seen[1] = 0;
            }
            const int first = seen[0] ? (int)__builtin_ctzll(seen[0]) >> 2 : 16 + ((int)__builtin_ctzll(seen[1] | 1ull << 63) >> 2);
            const int last  = seen[1] ? 31 - ((int)__builtin_clzll(seen[1]) >> 2) : seen[0] ? 15 - ((int)__builtin_clzll(seen[0]) >> 2) : -1;
            walk_end = last < 0 ? 0 : min(n_steps, wave + last * DEC_WAVES + 1);
            if (first == 0 || last < 0) break;
            walk = wave + first * DEC_WAVES;
        }
        convert_q();
    } else if (!Q_FIRST && !DEEP) {
        if (wave < n_steps) issue(wave, S0{});
    }

    // (V8) where the pieces of this lane's V units go: read behind the first K/V request, needed when that has arrived
    auto read_places = [&]() __attribute__((always_inline)) {
        if (!V8) return;
        static_assert(!V8 || (V8Places<D>::RAWSZ == RAWSZ && V8Places<D>::UNITS == NU * 64 && V8Places<D>::UNIT == UNIT), "table layout");
        const uint32_t * places = (const uint32_t *)v8_places_table<D>.at;
#pragma unroll
        for (int i = 0; i < NU; i++)
#pragma unroll
            for (int k = 0; k < PCS / 2; k++) vdst[i][k] = places[(i * 64 + lane) * (PCS / 2) + k];
    };
    typedef std::integral_constant<int, ONE ? 0 : 1> S1;
    auto walk_steps = [&]() __attribute__((always_inline)) {
        for (int it = walk; it < walk_end; it += 2 * DEC_WAVES) {
            step(it, it + DEC_WAVES, S0{});
            if (it + DEC_WAVES < walk_end) step(it + DEC_WAVES, it + 2 * DEC_WAVES, S1{});
        }
    };
    if constexpr (DEEP) {
        // (Pairs of steps, an odd one ahead of them out of stage 1, and one way out of the loop: a way past a pair's second step would
        //  make its rows uncountable again.)
        const int own = n_steps > wave ? (n_steps - wave + DEC_WAVES - 1) / DEC_WAVES : 0;        // the wave's steps
        int       it  = wave;
        request_q();                               // (ahead of K and V: it is converted while they are on their way)
        if (D == 128 || own <= 1) {                // (128-wide: ranges of one step a wave, see deep_rows)
            if (own >= 1) {
                issue(it, S0{});
                __builtin_amdgcn_sched_barrier(0);
                convert_q();
                step(it, -1, S0{});
            }
        } else {
            if (own & 1) {
                issue(it, S1{});
                issue(it + DEC_WAVES, S0{});
                __builtin_amdgcn_sched_barrier(0);
                convert_q();
                step(it, it + 2 * DEC_WAVES, S1{});
                it += DEC_WAVES;
            } else {
                issue(it, S0{});
                issue(it + DEC_WAVES, S1{});
                __builtin_amdgcn_sched_barrier(0);
                convert_q();
            }
            // (the last pair stands by itself: requests for no step are not free. 256 keys, 8 rows x 16 heads of 64 4.50 -> 4.31 us, 384, one row x 8,
            //  4.77 -> 4.56)
            while (it + 2 * DEC_WAVES < n_steps) {
                step(it, it + 2 * DEC_WAVES, S0{});
                step(it + DEC_WAVES, it + 3 * DEC_WAVES, S1{});
                it += 2 * DEC_WAVES;
            }
            step(it, -1, S0{});
            step(it + DEC_WAVES, -1, S1{});
        }
    } else if constexpr (Q_FIRST && !MASK) {
        // (Q ahead of K and V, whose request takes no branch of its own: it is converted while they are on their way.  Waves without a step ask
        //  for nothing: from empty buffers they kept the others' requests waiting, 5 rows x 32 query and 8
        //  KV heads of 128 against 28 Q8_0 entries 5.4 and 4.85 us, against 90 5.9 and 5.7)
        if (wave < n_steps) {
            request_q();
            issue(wave, S0{});
            read_places();
            convert_q();
            walk_steps();
        }
    } else {
        read_places();
        if (!MASK) {                               // (after the first K/V request: the two cold misses overlap)
            request_q();
            convert_q();
        }
        walk_steps();
    }

    // ---- column totals, then the four waves through LDS ----------------------------------------------
    l += xor_shuffle(l, 16);
    l += xor_shuffle(l, 32);
    if (!have) m = -INFINITY;
    __syncthreads();                           // every wave is done with its stage
#pragma unroll
    for (int db = 0; db < DBK; db++) *(float4v *)&red_o[wave][j][db * 16 + g4 * 4] = oacc[db];
    if (g4 == 0) {
        red_ml[wave][j][0] = m;
        red_ml[wave][j][1] = l;
    }
    __syncthreads();

    // thread t: column t / 16, D / 64 groups of four d
    const int col = tid >> 4;
    bool bad = false;                           // this column's result is not finite
    if (row0 + col < R) {
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; w++) M = fmaxf(M, red_ml[w][col][0]);
        float f[DEC_WAVES];
        float L = 0.0f;
#pragma unroll
        for (int w = 0; w < DEC_WAVES; w++) {
            const float mw = red_ml[w][col][0];
            f[w] = mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
            L += red_ml[w][col][1] * f[w];
        }
        bad = not_finite(L);
        const float den = L == 0.0f ? INFINITY : L;             // (a sum of NaN makes the row NaN, as on the CPU)
        const int     ciq1 = query_of(row0 + col);
        const int     ch   = hk * a.gqa + row0 + col - ciq1 * a.gqa;
        const int64_t row  = ((int64_t)b * a.Nq + ciq1) * a.Hq + ch;
        const int dv = PAD ? a.Dv : D;              // dst rows are dv floats; partial rows stay D apart
#pragma unroll
        for (int k = 0; k < D / 64; k++) {
            const int d = ((tid & 15) + k * 16) * 4;
            if (PAD && d >= dv) continue;
            float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < DEC_WAVES; w++) {
                const float4v o = *(const float4v *)&red_o[w][col][d];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] += o[e] * f[w];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) bad = bad || not_finite(acc[e]);
            if (a.n_splits == 1) {
                float4v o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = acc[e] / den;
                *(float4v *)(a.dst + row * dv + d) = o;
            } else {
                float * pa = a.part_acc + (row * a.n_splits + split) * D + d;
                if (a.counters) {
                    device_store2(pa, acc[0], acc[1]);
                    device_store2(pa + 2, acc[2], acc[3]);
                } else {
                    *(float4v *)pa = acc;
                }
            }
        }
        if (a.n_splits > 1 && (tid & 15) == 0) {
            // natural-log units, as the merge expects them
            float * pm = a.part_ml + (row * a.n_splits + split) * 2;
            const float mn = M == -INFINITY ? (L == L ? -INFINITY : 0.0f) : M * 0.6931471805599453f;      // (nor does the merge leave it out)
            if (a.counters) {
                device_store2(pm, mn, L);
            } else {
                pm[0] = mn;
                pm[1] = L;
            }
        }
    }
    // An excluded key was multiplied by a probability of zero above, not skipped.  For finite K/V that is the same thing; a
    // cache slot that holds NaN or inf bits (never written, and masked out for that reason) turns the products into NaN.
    // Such a row shows in its result, and is computed again the way the CPU op does it - excluded keys not read at all.
    // Without a mask every key is visible and a non-finite result is the answer.  (Columns 4w .. 4w + 3 belong to wave w
    // in both passes: the second store follows the first in the same wave.)
    bool redone = false;
    if constexpr (MASK) {
        const uint64_t badmask = __builtin_amdgcn_ballot_w64(bad);
        if (badmask != 0) {
            redone = true;
            __threadfence();
#pragma unroll 1
            for (int c = 0; c < 4; c++) {
                const int r = row0 + wave * 4 + c;
                if (((badmask >> (16 * c)) & 0xFFFFu) != 0 && r < R)
                    attn_row_redo<TYPE, D>(a, r / a.gqa, hk * a.gqa + r % a.gqa, b, split, k_begin, k_end);
            }
        }
    }
    // the last of the n_splits workgroups of this (chunk, KV head, batch) merges its rows: no launch for the merge
    if (a.n_splits > 1 && a.counters) {
        if (!fattn_last_of_set(a, set, a.n_splits, (int *)smem, redone)) return;
        constexpr int LPR = D / 4;                  // lanes per row: 8 or 4 rows per pass
        for (int c = tid / LPR; c < 16 && row0 + c < R; c += DEC_THREADS / LPR) {
            const int r = row0 + c;
            const int riq = query_of(r);
            fattn_merge_row<true>(a, ((int64_t)b * a.Nq + riq) * a.Hq + hk * a.gqa + r - riq * a.gqa, tid % LPR);
        }
    }
}

template <int D, int TYPE, bool MASK, bool RAW, bool V8, bool PAD = false>
__global__ void __launch_bounds__(DEC_THREADS) __attribute__((amdgpu_waves_per_eu((decode_waves_min<D, TYPE, RAW>()), (decode_waves_max<D, RAW, V8>()))))
fattn_decode_kernel(const FattnArgs a) {
    decode_body<D, TYPE, MASK, RAW, V8, PAD, false>(a, 0);
}

template <int D, bool MASK, int TYPE, bool RAW, bool V8, bool PAD, bool DEEP = false>
__device__ __forceinline__ void decode_short(const DecodeShort & p) {
    FattnArgs a = decode_expand(p, D);
    if (!PAD) a.Dv = D;
    decode_body<D, TYPE, MASK, RAW, V8, PAD, true, DEEP>(a, MASK ? (int)(p.Dv >> 16) : 0);
}
template <int D, int TYPE, bool RAW, bool V8, bool PAD>
__global__ void __launch_bounds__(DEC_THREADS) __attribute__((amdgpu_waves_per_eu((decode_waves_min<D, TYPE, RAW>()), (decode_waves_max<D, RAW, V8>()))))
fattn_decode_short_masked_kernel(const DecodeShort p) {
    decode_short<D, true, TYPE, RAW, V8, PAD>(p);
}

// Without a mask the requests of K, V and Q are made from the head of the arguments, ahead of the answer to the rest's: us a call in a
// stream, 20 heads of 64 against 1500, one row 6.50 -> 6.27, five 6.65 -> 6.44, 8 heads of 128 against 700 6.77 -> 6.57.  A mask's look
// and values need the tail's addresses; asked for behind K and V, or with the same head, those calls take 1 to 3% more than with a
// structure (8 sequences of 300 to 1000 entries 14.05 and 14.35 us, 32 of Q4_0 28.9 and 29.95).
// (64-wide f16 rows: 128 registers instead of 138, for four waves a SIMD, which pays where workgroups share a CU and walk long ranges; with
//  DEEP three waves, see deep_rows.)
template <int D, int TYPE, bool RAW, bool V8, bool PAD, bool DEEP>
__global__ void __launch_bounds__(DEC_THREADS)
__attribute__((amdgpu_waves_per_eu((D == 64 && TYPE == MI355X_TYPE_F16 ? (DEEP ? 3 : 4) : decode_waves_min<D, TYPE, RAW>()), (decode_waves_max<D, RAW, V8>()))))
fattn_decode_short_kernel(FATTN_HEAD_PARAMS, const ArgTail<DecodeShort> tail) {
    decode_short<D, false, TYPE, RAW, V8, PAD, DEEP>(fattn_join<DecodeShort>(FATTN_HEAD_ARGS, tail));
}

// Unmasked f16 rows: DEEP, but for 64-wide heads where the CUs' fourth workgroups, which its registers do not leave room for, would be a
// round of their own; on 128-wide heads, where two steps' rows take more registers than there are, ranges of one step a wave.
// us a call inside a graph, without and with it: 5 rows x 20 heads of 64 against 1500 6.96 -> 6.85, against 375, 8 heads, 5.88 -> 5.40,
// 64 sequences x 20 heads against 1500 77.0 -> 74.1 (1280 workgroups, two rounds either way), 8 sequences x 16 heads against 4000 27.4 ->
// 28.8 where its three workgroups a CU cost a round (so not taken); 16 heads of 80 x 5 rows 8.2 -> 7.8; 128-wide, 8 KV heads: 663 entries
// 7.1 -> 6.7, 2047 8.5 -> 8.0, 64 4.4 -> 4.1; with steps in pairs, spilling, 4000 10.2 -> 12.7, as taken 10.1.
static inline bool deep_rows(int D, int64_t wgs, int n_cus, int keys_per_split) {
    if (D == 128) return keys_per_split <= DEC_WAVES * STEP;
    return (wgs + 3 * n_cus - 1) / (3 * n_cus) == (wgs + 4 * n_cus - 1) / (4 * n_cus);
}

// the form of the kernel that a call takes; p: its arguments where they are short
template <int D, int TYPE, bool RAW, bool V8>
int form_of(const FattnArgs & a, DecodeShort & p) {
    if constexpr (TYPE == MI355X_TYPE_F16 || V8 || (RAW && TYPE != MI355X_TYPE_Q8_0)) {      // (the rows of a cache as they usually lie)
        if (decode_shorten(a, p))
            return TYPE == MI355X_TYPE_F16 && !a.mask && deep_rows(D, (int64_t)a.n_splits * a.Hkv * a.B, a.n_cus, a.n_splits > 1 ? a.keys_per_split : a.Nkv)
                       ? MI355X_FATTN_FORM_DEEP
                       : MI355X_FATTN_FORM_SHORT;
    }
    return MI355X_FATTN_FORM_GENERAL;
}

template <int D, int TYPE, bool MASK, bool RAW, bool V8 = false, bool PAD = false>
int launch_one(FattnArgs a, hipStream_t stream) {
    const int64_t pairs = (int64_t)a.n_splits * a.Hkv * a.B;
    const int64_t wgs   = a.q_chunks == 1 ? pairs : (pairs + 7) / 8 * 8 * a.q_chunks;      // as the kernel numbers them
    if (wgs > 0x7fffffff || a.q_chunks != (a.Nq * a.gqa + 15) / 16) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs);
    constexpr int lds = decode_lds_bytes<D, TYPE, RAW, V8>();
    if constexpr (TYPE == MI355X_TYPE_F16 || V8 || (RAW && TYPE != MI355X_TYPE_Q8_0)) {
        DecodeShort p;
        const int   form = form_of<D, TYPE, RAW, V8>(a, p);
        if (form != MI355X_FATTN_FORM_GENERAL) {
            if (MASK) p.Dv |= decode_turns(a, TYPE == MI355X_TYPE_F16 ? D * 2 : D / 32 * raw_block_bytes<TYPE>()) << 16;
            static std::atomic<uint64_t> short_lds_allowed{0};
            const dim3 short_grid((unsigned)a.n_splits, (unsigned)a.Hkv, (unsigned)a.B);
            if constexpr (MASK) {
                const hipError_t e = fattn_allow_lds((const void *)fattn_decode_short_masked_kernel<D, TYPE, RAW, V8, PAD>, lds, short_lds_allowed);
                if (e != hipSuccess) return (int)e;
                fattn_launch(fattn_decode_short_masked_kernel<D, TYPE, RAW, V8, PAD>, short_grid, dim3(DEC_THREADS), lds, stream, p);
            } else {
                if constexpr (TYPE == MI355X_TYPE_F16) {
                    static_assert(lds <= 64 * 1024, "no attribute to raise");
                    if (form == MI355X_FATTN_FORM_DEEP) {
                        fattn_launch_head(fattn_decode_short_kernel<D, TYPE, RAW, V8, PAD, true>, short_grid, dim3(DEC_THREADS), lds, stream, p);
                        return (int)hipGetLastError();
                    }
                }
                const hipError_t e = fattn_allow_lds((const void *)fattn_decode_short_kernel<D, TYPE, RAW, V8, PAD, false>, lds, short_lds_allowed);
                if (e != hipSuccess) return (int)e;
                fattn_launch_head(fattn_decode_short_kernel<D, TYPE, RAW, V8, PAD, false>, short_grid, dim3(DEC_THREADS), lds, stream, p);
            }
            return (int)hipGetLastError();
        }
    }
    a.by_splits = fast_div((uint32_t)a.n_splits);
    a.by_chunks = fast_div((uint32_t)a.q_chunks);
    a.by_hkv    = fast_div((uint32_t)a.Hkv);
    a.by_gqa    = fast_div((uint32_t)a.gqa);
    a.by_bq     = fast_div((uint32_t)a.bq);
    a.by_hm     = fast_div((uint32_t)a.Hm);
    a.by_bm     = fast_div((uint32_t)a.Bm);
    static std::atomic<uint64_t> lds_allowed{0};
    const hipError_t e = fattn_allow_lds((const void *)fattn_decode_kernel<D, TYPE, MASK, RAW, V8, PAD>, lds, lds_allowed);
    if (e != hipSuccess) return (int)e;
    fattn_launch((fattn_decode_kernel<D, TYPE, MASK, RAW, V8, PAD>), grid, dim3(DEC_THREADS), lds, stream, a);
    return (int)hipGetLastError();
}

// go(RAW, V8) of a call over whole heads: quantised rows that are streamed, and whether V goes through its int8 stage
template <int D, int TYPE, typename F>
int by_rows(const FattnArgs & a, F go) {
    typedef std::true_type  Yes;
    typedef std::false_type No;
    if constexpr (FATTN_IS_BLOCK_TYPE(TYPE)) {
        // contiguous rows, and every step of every (head, batch, split) starts on a unit boundary
        constexpr int RS   = D / 32 * raw_block_bytes<TYPE>();
        constexpr int UNIT = RS % 8 == 0 ? 8 : 4;
        const bool raw = a.nbk1 == RS && a.nbv1 == RS &&
                         !((uintptr_t)a.k % UNIT) && !((uintptr_t)a.v % UNIT) &&
                         !(a.nbk2 % UNIT) && !(a.nbk3 % UNIT) && !(a.nbv2 % UNIT) && !(a.nbv3 % UNIT);
        static const bool no_raw = getenv("MI355X_FATTN_DECODE_NO_STREAM") != nullptr;      // the per-lane path, for comparison runs
        if (raw && !no_raw) {
            if constexpr (TYPE == MI355X_TYPE_Q8_0) {
                static const bool f16_stage = getenv("MI355X_FATTN_DECODE_F16_STAGE") != nullptr;     // the earlier V path, for comparison runs
                if (!f16_stage) return go(Yes{}, Yes{});
            }
            return go(Yes{}, No{});
        }
    }
    return go(No{}, No{});
}

template <int D, int TYPE>
int launch(const FattnArgs & a, hipStream_t stream) {
    if (a.Dv != a.D) {              // another head size on f16 rows, or nothing
        if constexpr (TYPE == MI355X_TYPE_F16)
            return a.mask ? launch_one<D, TYPE, true, false, false, true>(a, stream) : launch_one<D, TYPE, false, false, false, true>(a, stream);
        return (int)hipErrorInvalidValue;
    }
    return by_rows<D, TYPE>(a, [&](auto raw, auto v8) {
        return a.mask ? launch_one<D, TYPE, true, raw(), v8()>(a, stream) : launch_one<D, TYPE, false, raw(), v8()>(a, stream);
    });
}
template <int D, int TYPE>
int form(const FattnArgs & a) {
    DecodeShort p;
    return by_rows<D, TYPE>(a, [&](auto raw, auto v8) { return form_of<D, TYPE, raw(), v8()>(a, p); });
}

}  // namespace

bool fattn_decode_supported(const FattnArgs & a, int ktype) {
    if (a.D != 64 && a.D != 128) return false;
    if (a.Dv != a.D && (a.Dv % 8 || a.Dv > a.D || ktype != MI355X_TYPE_F16)) return false;       // other head sizes: f16 rows read in place
    if (a.Nq < 1 || a.Nkv < 1) return false;
    if ((int64_t)a.Nq * a.gqa > ((int64_t)1 << 20)) return false;      // 16-row chunks of the rows that share a KV head
    if (a.softcap != 0.0f) return false;
    if (ktype == MI355X_TYPE_F16) return a.kv_aligned16 != 0;
    if (ktype == MI355X_TYPE_Q8_0) return a.kv_aligned4 != 0;
    if (FATTN_IS_BLOCK_TYPE(ktype)) return a.kv_aligned2 != 0;
    return false;
}

int fattn_decode_launch(const FattnArgs & a, int ktype, hipStream_t stream) {
    switch (ktype) {
#define DEC(T) case T: return a.D == 64 ? launch<64, T>(a, stream) : launch<128, T>(a, stream)
        DEC(MI355X_TYPE_F16);
        DEC(MI355X_TYPE_Q8_0);
        DEC(MI355X_TYPE_Q4_0);
        DEC(MI355X_TYPE_Q4_1);
        DEC(MI355X_TYPE_Q5_0);
        DEC(MI355X_TYPE_Q5_1);
#undef DEC
        default: return (int)hipErrorInvalidValue;
    }
}

int fattn_decode_form(const FattnArgs & a, int ktype) {
    switch (ktype) {
#define DEC(T) case T: return a.D == 64 ? form<64, T>(a) : form<128, T>(a)
        DEC(MI355X_TYPE_F16);
        DEC(MI355X_TYPE_Q8_0);
        DEC(MI355X_TYPE_Q4_0);
        DEC(MI355X_TYPE_Q4_1);
        DEC(MI355X_TYPE_Q5_0);
        DEC(MI355X_TYPE_Q5_1);
#undef DEC
        default: return MI355X_FATTN_FORM_GENERAL;
    }
}
