// The narrow forms of the copy kernels' arguments: which copies and SET_ROWS have one, and how a kernel walks it.  Nothing here
// touches a tensor's data (a test holds the walk, run on the CPU, to the tensors' own extents and strides).
#pragma once

#include "fattn_common.h"

#include <stddef.h>

// The two forms a copy's arguments take.  Narrow: both sides walked by the same (at most) four counts, units of dimension 0
// contiguous, spans below 4 GiB - what every cache write and read of the runtimes comes down to once adjacent dimensions that
// lie behind one another are one.  It is what it is because of its size: a launch whose kernel arguments take more than 112
// bytes costs the host 0.8 us more, 2 us on an idle queue (measured, bytes against us a launch in a chain of empty kernels: 16
// 2.5, 64 2.6, 112 2.7, 120 3.5, 352 3.7), and the 60 copies of a decoder step were bound by that.  Wide: everything else.
struct NarrowCopy {
    const char * src;
    char *       dst;
    int64_t      mirror;
    uint32_t     n;                        // units
    FastDiv      div[3];
    uint32_t     snb[3], dnb[3];           // pitches of counts 1 .. 3
    uint32_t     whole;                    // see whole_pieces
    typedef uint32_t index, offset;
};
static_assert(sizeof(NarrowCopy) <= 112, "arguments of a cheap launch");

// The same with all that the loads' addresses need in the first 56 bytes: one line of the scalar cache, which for a large copy can be in
// registers when its waves start (see ArgTail).  All kernels but the quantising ones read this order, whose second line is wanted for the
// stores alone.  us a copy in a graph, the order above and this one, rows x 8 heads of 128: from Q8_0 663 rows of 704 2.48, 2.30, 407 2.18, 2.02,
// 1500 of 2048 2.85, 2.68; Q8_0 as it is 663 2.37, 2.23; F32 to F16 128 2.05, 1.87, 407 2.38, 2.19; 8 x 300 rows of 37 2.17, 2.00.  Quantising
// copies have work enough behind their loads, and the shifts to be taken apart show: F32 to Q4_0 128 rows 2.13, 2.25, 407 2.50, 2.57.
struct NarrowCopyHead {
    const char * src;
    uint32_t     n;
    uint32_t     d[3], m[3], shifts;       // of div, a byte for each shift; the fourth byte: whole
    uint32_t     snb[3], dnb[3];
    char *       dst;
    int64_t      mirror;
    typedef uint32_t index, offset;
    template <typename F> __host__ __device__ void pointers(F f) { f(src, dst); }
};
static_assert(sizeof(NarrowCopyHead) <= 112 && offsetof(NarrowCopyHead, dnb) < 56, "arguments of a cheap launch");
static inline NarrowCopyHead head_first(const NarrowCopy & a) {
    NarrowCopyHead h = {a.src, a.n, {}, {}, a.whole << 24, {}, {}, a.dst, a.mirror};
    for (int i = 0; i < 3; i++) {
        h.d[i] = a.div[i].d;
        h.m[i] = a.div[i].m;
        h.shifts |= a.div[i].s << (8 * i);
        h.snb[i] = a.snb[i];
        h.dnb[i] = a.dnb[i];
    }
    return h;
}
static __host__ __device__ __forceinline__ NarrowCopy narrow_of(const NarrowCopyHead & h) {
    const uint32_t s = h.shifts;
    return {h.src, h.dst, h.mirror, h.n, {{h.d[0], h.m[0], s & 31}, {h.d[1], h.m[1], s >> 8 & 31}, {h.d[2], h.m[2], s >> 16 & 31}},
            {h.snb[0], h.snb[1], h.snb[2]}, {h.dnb[0], h.dnb[1], h.dnb[2]}, s >> 24};
}

// The same two forms for SET_ROWS: narrow where rows, indices and pitches need 32 bits and nothing is mirrored.  Broadcast
// indices have a pitch of zero in it (x1, x2: their pitches along dimensions 2 and 3).
struct NarrowRows {
    const char * src;
    char *       dst;
    const char * idx;
    uint32_t     n;                        // units
    FastDiv      div[3];
    uint32_t     snb[3], dnb[3];
    uint32_t     x0, x1, x2_is_i64;        // x2_is_i64: x2 in the upper 31 bits
    uint32_t     rows;                     // of the destination
    typedef uint32_t index;
};
static_assert(sizeof(NarrowRows) <= 112, "arguments of a cheap launch");

// unit i's place along the four counts
struct Units {
    uint32_t i0, i1, i2, i3;
};
static __host__ __device__ __forceinline__ Units units_of(uint32_t i, const FastDiv (&div)[3]) {
    const uint32_t r1 = divide(i, div[0]), r2 = divide(r1, div[1]), i3 = divide(r2, div[2]);
    return {i - r1 * div[0].d, r1 - r2 * div[1].d, r2 - i3 * div[2].d, i3};
}
// byte offsets of unit i on both sides; sstep and dstep: bytes from one unit to the next along dimension 0
static __host__ __device__ __forceinline__ void offsets(const NarrowCopy & a, uint32_t i, int, uint32_t sstep, uint32_t dstep, uint32_t & so, uint32_t & to) {
    const Units u = units_of(i, a.div);
    so = u.i0 * sstep + u.i1 * a.snb[0] + u.i2 * a.snb[1] + u.i3 * a.snb[2];
    to = u.i0 * dstep + u.i1 * a.dnb[0] + u.i2 * a.dnb[1] + u.i3 * a.dnb[2];
}
// of the source unit, of the destination's unit in row 0, of the row's index
static __host__ __device__ __forceinline__ void offsets(const NarrowRows & a, uint32_t i, uint32_t sstep, uint32_t dstep, uint32_t & so, uint32_t & to, uint32_t & xo) {
    const Units u = units_of(i, a.div);
    so = u.i0 * sstep + u.i1 * a.snb[0] + u.i2 * a.snb[1] + u.i3 * a.snb[2];
    to = u.i0 * dstep + u.i2 * a.dnb[1] + u.i3 * a.dnb[2];
    xo = u.i1 * a.x0 + u.i2 * a.x1 + u.i3 * (a.x2_is_i64 >> 1);
}

// bytes from a tensor's first to its last, dimension by dimension; false at 4 GiB (less one 16-byte access)
static bool add_span(int64_t & span, int64_t count, int64_t pitch) {
    constexpr int64_t top = ((int64_t)1 << 32) - 16;
    if (pitch < 0 || (pitch > 0 && count - 1 > (top - span) / pitch)) return false;
    span += (count - 1) * pitch;
    return true;
}

// One side of a copy as counts and pitches (bytes) in the order of its elements: counts of one left out, dimensions that lie
// behind one another joined.  step: bytes of a unit.
struct Walk {
    int     n;
    int64_t count[4], pitch[4];
};
static Walk walk_of(const int64_t (&ne)[4], const int64_t (&nb)[4], int64_t unit0, int64_t step) {
    Walk w;
    w.n = 0;
    for (int i = 0; i < 4; i++) {
        const int64_t c = i ? ne[i] : ne[0] / unit0, p = i ? nb[i] : step;
        if (c == 1) continue;
        if (w.n && p == w.count[w.n - 1] * w.pitch[w.n - 1]) {
            w.count[w.n - 1] *= c;
        } else {
            w.count[w.n] = c;
            w.pitch[w.n++] = p;
        }
    }
    return w;
}

// What the runs of a destination's units are whole pieces of, the end of a contiguous destination aside: 128-byte lines 2, 32-byte
// sectors 1, neither 0.
static int whole_pieces(const char * dst, const Walk & t, int64_t dstep) {
    const int first = t.n && t.pitch[0] == dstep ? 1 : 0;          // (units that lie behind one another)
    uint64_t  bits  = (uint64_t)(uintptr_t)dst;
    if (t.n > first) bits |= (uint64_t)(first ? t.count[0] * dstep : dstep);
    for (int i = first; i < t.n; i++) bits |= (uint64_t)t.pitch[i];
    return bits % 128 == 0 ? 2 : bits % 32 == 0 ? 1 : 0;
}

// The narrow form, where there is one: the two sides cut into the same counts, the first of them units that are adjacent on both.
static bool narrow_copy(const CpyArgs & a, int64_t unit0, int64_t sstep, int64_t dstep, int64_t threads, NarrowCopy & v) {
    if (threads + 256 >= ((int64_t)1 << 31)) return false;
    const Walk s = walk_of(a.sne, a.snb, unit0, sstep), t = walk_of(a.dne, a.dnb, unit0, dstep);
    int64_t count[4] = {1, 1, 1, 1}, sp[4] = {0, 0, 0, 0}, dp[4] = {0, 0, 0, 0};
    int64_t cs = s.n ? s.count[0] : 1, ps = s.n ? s.pitch[0] : 0, ct = t.n ? t.count[0] : 1, pt = t.n ? t.pitch[0] : 0;
    // (count 0 is the units': one of them where a row is a single unit)
    int k = s.n && (ps != sstep || pt != dstep) ? 1 : 0;
    for (int i = 0, j = 0; i < s.n && j < t.n;) {
        const int64_t c = cs < ct ? cs : ct;
        if (k == 4 || cs % c || ct % c) return false;
        count[k] = c;
        sp[k]    = ps;
        dp[k++]  = pt;
        if ((cs /= c) > 1) ps *= c;
        else if (++i < s.n) { cs = s.count[i]; ps = s.pitch[i]; }
        if ((ct /= c) > 1) pt *= c;
        else if (++j < t.n) { ct = t.count[j]; pt = t.pitch[j]; }
    }
    v.src    = a.src;
    v.dst    = a.dst;
    v.mirror = a.mirror;
    v.n      = (uint32_t)a.n;
    v.whole  = (uint32_t)whole_pieces(a.dst, t, dstep);
    int64_t sspan = sstep, dspan = dstep;
    sp[0] = sstep;
    dp[0] = dstep;
    for (int i = 0; i < 4; i++)
        if (!add_span(sspan, count[i], sp[i]) || !add_span(dspan, count[i], dp[i])) return false;
    for (int i = 0; i < 3; i++) {
        v.div[i] = fast_div((uint32_t)count[i]);
        v.snb[i] = (uint32_t)sp[i + 1];
        v.dnb[i] = (uint32_t)dp[i + 1];
    }
    return true;
}

// SET_ROWS likewise
static bool narrow_rows(const CpyArgs & a, int64_t unit0, int64_t threads, NarrowRows & v) {
    const int64_t top = (int64_t)1 << 31;
    if (threads + 256 >= top || a.mirror || a.snb[0] != 4 || a.dne[1] >= top || a.dnb[1] < 0 || a.dnb[1] >= top) return false;
    int64_t sspan = a.sne[0] * 4, dspan = a.sne[0] * 4, xspan = 8, x[3];        // (a row is not longer than its F32 source)
    for (int i = 0; i < 3; i++) {
        if (i && a.ine[i] != 1 && a.ine[i] != a.sne[i + 1]) return false;
        x[i] = i && a.ine[i] == 1 ? 0 : a.inb[i];
        const int64_t n = a.sne[i + 1];
        if (x[i] >= top || !add_span(sspan, n, a.snb[i + 1]) || (i && !add_span(dspan, n, a.dnb[i + 1])) || !add_span(xspan, n, x[i])) return false;
        v.div[i] = fast_div((uint32_t)(i ? a.sne[i] : a.sne[0] / unit0));
        v.snb[i] = (uint32_t)(n == 1 ? 0 : a.snb[i + 1]);
        v.dnb[i] = (uint32_t)(i && n == 1 ? 0 : a.dnb[i + 1]);
    }
    v.src  = a.src;
    v.dst  = a.dst;
    v.idx  = a.idx;
    v.n    = (uint32_t)a.n;
    v.x0   = (uint32_t)x[0];
    v.x1   = (uint32_t)x[1];
    v.x2_is_i64 = (uint32_t)x[2] << 1 | (uint32_t)(a.idx_is_i64 != 0);
    v.rows = (uint32_t)a.dne[1];
    return true;
}
