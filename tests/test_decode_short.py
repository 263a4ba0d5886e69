"""The decode kernel's short form of its arguments, on the CPU: what it takes, expanded again, names the same addresses, rows and ranges as
the wide form, and it leaves what does not fit."""
import os
import subprocess

import pytest

from crispasr_amd import build

PROGRAM = r"""
#include "decode_short.h"
#include <cstdio>
#include <cstdlib>
#include <random>

static std::mt19937_64 rng(7);
static int64_t pick(int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); }
#define CHECK(x) do { if (!(x)) { printf("%s, call %d\n", #x, call); return 1; } } while (0)

int main() {
    int taken = 0, left = 0;
    for (int call = 0; call < 200000; call++) {
        FattnArgs a = {};
        a.D = a.Dv = pick(0, 1) ? 64 : 128;
        if (pick(0, 9) == 0) a.Dv = a.D - 8;
        a.gqa = (int)pick(1, 8); a.Nq = (int)pick(1, 20); a.Hkv = (int)pick(1, pick(0, 20) ? 40 : 70000); a.Hq = a.Hkv * a.gqa;
        a.B = (int)pick(1, 9); a.Bk = pick(0, 1) ? a.B : pick(0, 3) ? 1 : a.B % 3 == 0 ? 3 : 1; a.bq = a.B / a.Bk;
        a.q_chunks = (a.Nq * a.gqa + 15) / 16;
        a.Nkv = (int)pick(1, 5000);
        a.n_splits = pick(0, 1) ? 1 : (int)pick(2, pick(0, 9) ? 20 : 256);
        a.keys_per_split = a.n_splits == 1 ? a.Nkv : (a.Nkv + a.n_splits - 1) / a.n_splits;
        if (a.n_splits > 1 && pick(0, 9)) a.keys_per_split = (a.keys_per_split + 31) / 32 * 32;
        auto stride = [&]() { return pick(0, 30) ? pick(0, 1 << 20) * 2 : pick(0, 30) ? (int64_t)4294967290 : (int64_t)1 << 33; };
        a.nbq1 = stride(); a.nbq2 = stride(); a.nbq3 = stride();
        a.nbk1 = a.nbv1 = stride(); a.nbk2 = a.nbv2 = stride(); a.nbk3 = a.nbv3 = stride();
        if (pick(0, 9) == 0) a.nbv2 += 64;
        if (pick(0, 9) == 0) a.nbv3 += 64;
        a.nbm1 = stride(); a.nbm2 = stride(); a.nbm3 = stride();
        a.Hm = pick(0, 1) ? 1 : pick(0, 4) ? a.Hq : a.gqa; a.Bm = pick(0, 1) ? 1 : a.B;
        a.q = (const char *)0x1000000000; a.k = a.q + 4096; a.v = a.q + 8192; a.mask = pick(0, 1) ? a.q + 64 : nullptr; a.masked = a.mask != nullptr;
        a.dst = (float *)(a.q + 128); a.scale = 0.25f; a.max_bias = pick(0, 9) ? 0.0f : 8.0f; a.softcap = pick(0, 9) ? 0.0f : 30.0f;
        a.part_acc = (float *)(a.q + 256); a.part_ml = a.part_acc + (int64_t)a.Nq * a.Hq * a.B * a.n_splits * a.D + (pick(0, 20) ? 0 : 4);
        a.counters = pick(0, 1) ? (unsigned *)(a.q + 512) : nullptr;
        DecodeShort p;
        if (!decode_shorten(a, p)) { left++; continue; }
        taken++;
        const FattnArgs e = decode_expand(p, a.D);
        CHECK(a.max_bias <= 0.0f && a.softcap == 0.0f && a.Nq * a.gqa <= 16);
        CHECK(e.q == a.q && e.k == a.k && e.v == a.v && e.mask == a.mask && e.dst == a.dst && e.scale == a.scale && e.masked == a.masked);
        CHECK(e.D == a.D && e.Dv == a.Dv && e.Nq == a.Nq && e.gqa == a.gqa && e.Hq == a.Hq && e.Hkv == a.Hkv && e.B == a.B && e.Nkv == a.Nkv);
        CHECK(e.n_splits == a.n_splits && e.keys_per_split == a.keys_per_split);
        if (a.n_splits > 1) CHECK(e.part_acc == a.part_acc && e.part_ml == a.part_ml && e.counters == a.counters);
        for (int t = 0; t < 8; t++) {
            const int64_t b = pick(0, a.B - 1), h = pick(0, a.Hq - 1), i = pick(0, a.Nq - 1), j = pick(0, a.Nkv - 1);
            CHECK(i * e.nbq1 + h * e.nbq2 + b * e.nbq3 == i * a.nbq1 + h * a.nbq2 + b * a.nbq3);
            CHECK(j * e.nbk1 + h / e.gqa * e.nbk2 + b / e.bq * e.nbk3 == j * a.nbk1 + h / a.gqa * a.nbk2 + b / a.bq * a.nbk3);
            CHECK(j * e.nbv1 + h / e.gqa * e.nbv2 + b / e.bq * e.nbv3 == j * a.nbv1 + h / a.gqa * a.nbv2 + b / a.bq * a.nbv3);
            // (the kernel's own: head and sequence times their strides; and what the row loop makes of Hm and Bm)
            if (a.mask) CHECK(i * e.nbm1 + h * e.nbm2 + b * e.nbm3 == i * a.nbm1 + h % a.Hm * a.nbm2 + b % a.Bm * a.nbm3);
            if (a.mask) CHECK(i * e.nbm1 + h % e.Hm * e.nbm2 + b % e.Bm * e.nbm3 == i * a.nbm1 + h % a.Hm * a.nbm2 + b % a.Bm * a.nbm3);
        }
        // the kernel divides rows by gqa in f32, with a reciprocal that may be an ulp off
        for (int row = 0; row < 16; row++)
            for (int off = -1; off <= 1; off++) {
                union { float f; uint32_t u; } r = {1.0f / (float)a.gqa};
                r.u += (uint32_t)off;
                CHECK((int)(((float)row + 0.5f) * r.f) == row / a.gqa);
            }
    }
    printf("taken %d left %d\n", taken, left);
    return taken > 10000 && left > 10000 ? 0 : 2;
}
"""


def test_short_arguments(tmp_path):
    if not os.path.exists(build._hipcc()):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    flags = ["--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", "-I", build.CSRC]
    res = subprocess.run([build._hipcc(), *flags, str(src), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr[-3000:]
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
