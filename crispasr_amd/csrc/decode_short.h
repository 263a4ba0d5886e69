// The decode kernel's arguments in 112 bytes (internal).  With them a workgroup finds its place without a division and has half the
// scalar loads ahead of its first request; calls inside a graph, us, 376 bytes and these: 5 rows x 20 heads of 64 against 560
// masked entries 6.95 -> 6.27, against 1500 7.0 -> 6.8, 8 heads of 128 against 2048 masked Q8_0 entries 9.1 -> 8.55, 663 entries
// 7.4 -> 7.25.  A launch also costs the host 0.9 us less than one with 376 bytes (three launches of which one does 9.4 -> 8.5 us).
#pragma once

#include "fattn_common.h"

#include <stddef.h>

// A step's call as the runtimes make it: up to 16 rows per KV head, K and V alike in their strides, no slopes, a mask that is one
// head's or every head's own and one sequence's or every sequence's own.  Extents that one value stands for have a stride of zero.
// The first requests of K, V and Q come from the first 56 bytes (see ArgTail).
struct DecodeShort {
    const char * k;
    const char * v;
    const char * q;
    uint32_t     nbk1, nbk2, nbk3;    // and V's
    uint32_t     nbq1, nbq2, nbq3;
    uint32_t     Nkv;
    uint32_t     rows;                // Nq | gqa << 5 | n_splits << 10 | keys_per_split / 32 << 17 (0: not cut)
    const char * mask;
    uint32_t     nbm1, nbm2, nbm3;
    uint32_t     heads;               // Hkv | B << 16
    float        scale;
    uint32_t     Dv;                  // | sequences in the first round << 16 (0: in their own order, see decode_turns)
    float *      dst;
    float *      part_acc;            // the (max, sum) pairs lie right behind it
    unsigned *   counters;
    template <typename F> __host__ __device__ void pointers(F f) { f(k, v, q, mask, dst, part_acc, counters); }
};
static_assert(sizeof(DecodeShort) == 112 && offsetof(DecodeShort, mask) == 56, "see above");

// Sequences of different lengths in one call (a mask of every sequence's own ends each), more workgroups than CUs: a CU that gets the
// workgroups of two long ones is the last.  Workgroup n_cus + i comes to the CU of workgroup i, so the sequences of the first round (a
// workgroup on every CU) go in their own order, and those behind them by length (sequence_of_turn): the longest beside the shortest.
// In graphs, 32 query, 8 KV heads of 128, lengths spread evenly and shuffled, us: 64 sequences of 500 to 4096 Q8_0 entries 81 -> 71, of
// 200 to 2048 f16 entries 69 -> 55, 40 of these 64 -> 52, 128 of 300 to 2048 Q8_0 entries 77 -> 68, 64 of 100 to 512 16.9 -> 15.9;
// of one length 99.9 -> 99.9 (4096), 19.6 -> 19.6 (36 x 600).  (The first round by length as well, from the middle to the longest, is
// better yet where few CUs get a second workgroup, 40 f16 sequences 44, but its look is in nobody's shadow: +1.2 us.)
// Not where the look has nothing to hide behind: below 64 kB of a head's K (64 sequences of 512 Q8_0 entries have 70), and for rows that
// are bound by their dequantising (all but f16 and Q8_0 of 128) below 128 kB and where the second round is not whole: 48 sequences of
// 1000 Q4_0 entries 24.1 -> 25.1, of 2048 Q8_0 entries of 64 26.4 -> 27.2; 64 of 400 to 4000 Q4_0 entries of 64 44.3 -> 42.5.
// Returns the sequences in the first round, or 0: their own order.
static inline uint32_t decode_turns(const FattnArgs & a, int row_bytes) {
    if (!a.mask || a.n_splits != 1 || a.Bm != a.B || a.B < 2 || a.B > 128 || a.Hkv > a.n_cus || (int64_t)a.Hkv * a.B <= a.n_cus) return 0;
    const int  first = a.n_cus / a.Hkv;            // (below B)
    const bool wide  = row_bytes >= 128;
    if ((int64_t)a.Nkv * row_bytes < (wide ? 64 : 128) * 1024 || (!wide && a.B < 2 * first)) return 0;
    return (uint32_t)first;
}

// false: the call needs the wide form
static inline bool decode_shorten(const FattnArgs & a, DecodeShort & p) {
    const int64_t nb[12] = {a.nbq1, a.nbq2, a.nbq3, a.nbk1, a.nbk2, a.nbk3, a.nbv1, a.nbv2, a.nbv3, a.nbm1, a.nbm2, a.nbm3};
    for (int i = 0; i < (a.mask ? 12 : 9); i++)
        if ((uint64_t)nb[i] > 0xFFFFFFFFull) return false;
    if (a.nbk1 > 1 << 26) return false;                       // (32 rows are within 4 GiB)
    const bool    one_sequence = a.Bk == 1;
    const int64_t rows = (int64_t)a.Nq * a.Hq * a.B;
    if (a.q_chunks != 1 || a.Nq < 1 || a.gqa < 1 || (int64_t)a.Nq * a.gqa > 16 || a.max_bias > 0.0f || a.softcap != 0.0f) return false;
    if (!(one_sequence || a.Bk == a.B) || a.nbk1 != a.nbv1 || a.nbk2 != a.nbv2 || (!one_sequence && a.nbk3 != a.nbv3)) return false;
    if (a.mask && (!(a.Hm == 1 || a.Hm == a.Hq) || !(a.Bm == 1 || a.Bm == a.B))) return false;
    if (a.Hkv > 0xFFFF || a.B > 0xFFFF || a.Hq != a.Hkv * a.gqa) return false;
    if (a.n_splits > 127 || (a.n_splits > 1 && (a.keys_per_split % 32 || a.keys_per_split / 32 < 1 || a.keys_per_split / 32 > 0x7FFF))) return false;
    if (a.n_splits > 1 && a.part_ml != a.part_acc + rows * a.n_splits * a.D) return false;
    if (a.n_splits == 1 && a.keys_per_split < a.Nkv) return false;
    p.q = a.q; p.k = a.k; p.v = a.v; p.mask = a.mask; p.dst = a.dst;
    p.part_acc = a.n_splits > 1 ? a.part_acc : nullptr;
    p.counters = a.n_splits > 1 ? a.counters : nullptr;
    p.nbq1 = (uint32_t)a.nbq1; p.nbq2 = (uint32_t)a.nbq2; p.nbq3 = (uint32_t)a.nbq3;
    p.nbk1 = (uint32_t)a.nbk1; p.nbk2 = (uint32_t)a.nbk2; p.nbk3 = one_sequence ? 0 : (uint32_t)a.nbk3;
    p.nbm1 = a.mask ? (uint32_t)a.nbm1 : 0;
    p.nbm2 = a.mask && a.Hm > 1 ? (uint32_t)a.nbm2 : 0;
    p.nbm3 = a.mask && a.Bm > 1 ? (uint32_t)a.nbm3 : 0;
    p.scale = a.scale;
    p.Nkv   = (uint32_t)a.Nkv;
    p.rows  = (uint32_t)a.Nq | (uint32_t)a.gqa << 5 | (uint32_t)a.n_splits << 10 | (a.n_splits > 1 ? (uint32_t)(a.keys_per_split / 32) << 17 : 0);
    p.heads = (uint32_t)a.Hkv | (uint32_t)a.B << 16;
    p.Dv    = (uint32_t)a.Dv;
    return true;
}

// what the kernel reads of the wide form (a stride of zero for the extents that one value stands for)
static __host__ __device__ __forceinline__ FattnArgs decode_expand(const DecodeShort & p, int D) {
    FattnArgs a = {};
    a.q = p.q; a.k = p.k; a.v = p.v; a.mask = p.mask; a.dst = p.dst;
    a.D  = D;
    a.Dv = (int)(p.Dv & 0xFFFFu);
    a.Nq = (int)(p.rows & 31u);
    a.gqa = (int)(p.rows >> 5 & 31u);
    a.n_splits = (int)(p.rows >> 10 & 127u);
    a.Nkv = (int)p.Nkv;
    a.keys_per_split = a.n_splits > 1 ? (int)(p.rows >> 17) * 32 : a.Nkv;
    a.Hkv = (int)(p.heads & 0xFFFFu);
    a.B = a.Bk = (int)(p.heads >> 16);
    a.Hq = a.Hkv * a.gqa;
    a.bq = a.q_chunks = 1;
    a.Hm = p.nbm2 ? a.Hq : 1;
    a.Bm = p.nbm3 ? a.B : 1;
    a.masked = p.mask != nullptr;
    a.nbq1 = p.nbq1; a.nbq2 = p.nbq2; a.nbq3 = p.nbq3;
    a.nbk1 = a.nbv1 = p.nbk1; a.nbk2 = a.nbv2 = p.nbk2; a.nbk3 = a.nbv3 = p.nbk3;
    a.nbm1 = p.nbm1; a.nbm2 = p.nbm2; a.nbm3 = p.nbm3;
    a.scale = p.scale;
    a.part_acc = p.part_acc;
    a.part_ml  = p.part_acc + (int64_t)a.Nq * a.Hq * a.B * a.n_splits * D;
    a.counters = p.counters;
    return a;
}
