"""The narrow form of a copy's arguments (counts, pitches and 32-bit offsets that both sides share) against the tensors' own extents
and strides, unit by unit, on the CPU: every shape, order and stride that the rule takes walks exactly the elements, in their order,
that the general form walks, and the rule leaves what needs more than 32 bits."""
import os
import subprocess

import pytest

from crispasr_amd import build

PROGRAM = r"""
#include "copy_forms.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

static std::mt19937_64 rng(20);
static int64_t pick(int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); }
static int64_t small() { static const int64_t c[] = {1, 1, 2, 3, 4, 6, 8, 12, 16, 24}; return c[rng() % 10]; }

// offset of unit i by definition
static int64_t at(const int64_t (&ne)[4], const int64_t (&nb)[4], int64_t unit0, int64_t step, int64_t i) {
    const int64_t n0 = ne[0] / unit0;
    return i % n0 * step + i / n0 % ne[1] * nb[1] + i / n0 / ne[1] % ne[2] * nb[2] + i / n0 / ne[1] / ne[2] * nb[3];
}

// strides of dense memory in some order of the dimensions, with gaps, overlaps (a pitch of zero) or pitches beyond 32 bits here and there
static void strides(const int64_t (&ne)[4], int64_t (&nb)[4], int64_t unit0, int64_t es, int64_t step) {
    int order[4] = {0, 1, 2, 3};
    if (rng() % 2) for (int i = 3; i > 1; i--) std::swap(order[i], order[1 + rng() % i]);
    nb[0] = es;
    int64_t next = ne[0] / unit0 * step;
    for (int k = 1; k < 4; k++) {
        if (rng() % 4 == 0) next += step * pick(1, 5);
        nb[order[k]] = next;
        next *= ne[order[k]];
    }
    if (rng() % 8 == 0) nb[pick(1, 3)] = 0;
    if (rng() % 8 == 0) nb[pick(1, 3)] = ((int64_t)1 << pick(29, 34)) + step * pick(0, 9);
}

int main() {
    long narrow = 0, wide = 0, reshaped = 0;
    for (int t = 0; t < 60000; t++) {
        CpyArgs a;
        memset(&a, 0, sizeof(a));
        const int64_t unit0 = rng() % 2 ? 32 : (int64_t)1 << pick(0, 3), sstep = unit0 * pick(1, 4), dstep = unit0 * pick(1, 4);
        int64_t n = 1;
        for (int i = 0; i < 4; i++) n *= a.sne[i] = i ? small() : unit0 * small();
        memcpy(a.dne, a.sne, sizeof(a.sne));
        if (rng() % 2) {                                  // another shape of as many units
            int64_t left = n / unit0;
            for (int i = 0; i < 4; i++) {
                int64_t c = i == 3 ? left : small();
                while (left % c) c--;
                a.dne[i] = i ? c : unit0 * c;
                left /= c;
            }
        }
        strides(a.sne, a.snb, unit0, sstep / unit0, sstep);
        strides(a.dne, a.dnb, unit0, dstep / unit0, dstep);
        a.n = n / unit0;
        NarrowCopy v;
        if (!narrow_copy(a, unit0, sstep, dstep, a.n, v)) { wide++; continue; }
        narrow++;
        reshaped += memcmp(a.sne, a.dne, sizeof(a.sne)) != 0;
        if ((int64_t)v.n != a.n) return printf("units %u %lld\n", v.n, (long long)a.n), 1;
        v.whole = (uint32_t)pick(0, 2);
        const NarrowCopy w = narrow_of(head_first(v));            // the order of the loads
        if (w.src != v.src || w.dst != v.dst || w.mirror != v.mirror || w.n != v.n || w.whole != v.whole || memcmp(w.div, v.div, sizeof(v.div)) ||
            memcmp(w.snb, v.snb, sizeof(v.snb)) || memcmp(w.dnb, v.dnb, sizeof(v.dnb)))
            return printf("copy %d: another order\n", t), 1;
        for (int64_t i = 0; i < a.n; i++) {
            uint32_t so, to;
            offsets(v, (uint32_t)i, (int)unit0, (uint32_t)sstep, (uint32_t)dstep, so, to);
            if (so != at(a.sne, a.snb, unit0, sstep, i) || to != at(a.dne, a.dnb, unit0, dstep, i) || to + dstep > ((int64_t)1 << 32))
                return printf("copy %d unit %lld: %u %u\n", t, (long long)i, so, to), 1;
        }
    }
    if (narrow < 20000 || wide < 2000 || reshaped < 2000) return printf("kinds %ld %ld %ld\n", narrow, wide, reshaped), 1;
    narrow = wide = 0;
    for (int t = 0; t < 40000; t++) {
        CpyArgs a;
        memset(&a, 0, sizeof(a));
        const int64_t unit0 = rng() % 2 ? 32 : rng() % 2 ? 8 : 1, dstep = unit0 * pick(1, 4);
        a.idx_is_i64 = rng() % 2;
        for (int i = 0; i < 4; i++) a.sne[i] = a.dne[i] = i ? small() : unit0 * small();
        a.dne[1] = rng() % 16 ? a.sne[1] + pick(0, 9) : ((int64_t)1 << pick(29, 33));
        strides(a.sne, a.snb, unit0, 4, unit0 * 4);
        strides(a.dne, a.dnb, unit0, 1, dstep);
        for (int i = 0; i < 3; i++) {
            a.ine[i] = i == 0 || rng() % 2 ? a.sne[i + 1] : 1;
            if (i && rng() % 8 == 0 && a.sne[i + 1] % 2 == 0) a.ine[i] = 2;
            a.inb[i] = (a.idx_is_i64 ? 8 : 4) * (i ? a.inb[i - 1] / 4 * a.ine[i - 1] : 1 + pick(0, 1));
            if (rng() % 16 == 0) a.inb[i] = (int64_t)1 << pick(29, 33);
        }
        a.mirror = rng() % 16 == 0 ? 4096 : 0;
        a.n = a.sne[0] / unit0 * a.sne[1] * a.sne[2] * a.sne[3];
        NarrowRows v;
        if (!narrow_rows(a, unit0, a.n, v)) { wide++; continue; }
        narrow++;
        if ((int64_t)v.n != a.n || a.mirror || (int64_t)v.rows != a.dne[1] || v.dnb[0] != a.dnb[1] || (v.x2_is_i64 & 1) != (uint32_t)a.idx_is_i64) return printf("rows %d\n", t), 1;
        for (int64_t i = 0; i < a.n; i++) {
            const int64_t n0 = a.sne[0] / unit0, i1 = i / n0 % a.sne[1], i2 = i / n0 / a.sne[1] % a.sne[2], i3 = i / n0 / a.sne[1] / a.sne[2];
            uint32_t so, to, xo;
            offsets(v, (uint32_t)i, (uint32_t)unit0 * 4, (uint32_t)dstep, so, to, xo);
            if (so != at(a.sne, a.snb, unit0, unit0 * 4, i) || to != i % n0 * dstep + i2 * a.dnb[2] + i3 * a.dnb[3] ||
                xo != i1 * a.inb[0] + i2 % a.ine[1] * a.inb[1] + i3 % a.ine[2] * a.inb[2])
                return printf("rows %d unit %lld: %u %u %u\n", t, (long long)i, so, to, xo), 1;
        }
    }
    if (narrow < 10000 || wide < 2000) return printf("kinds of rows %ld %ld\n", narrow, wide), 1;
    puts("ok");
    return 0;
}
"""


def test_narrow_forms_walk_what_the_tensors_say(tmp_path):
    if not os.path.exists(build._hipcc()):
        pytest.skip("no hipcc")
    src = tmp_path / "forms.cpp"
    src.write_text(PROGRAM)
    cmd = [build._hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I", build.CSRC, str(src), "-o", str(tmp_path / "forms")]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr[-3000:]
    res = subprocess.run([str(tmp_path / "forms")], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and res.stdout.endswith("ok\n"), res.stdout + res.stderr
