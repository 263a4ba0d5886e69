"""The fused rel-pos attention kernel at the ends of its walk: NaN bits behind the last key and on both sides of the table (views into longer
buffers), calls of one, two and more tiles, whose last step takes no products, tiles and whole sequences that the mask hides."""
import dataclasses

import numpy as np
import pytest

import oracle as ora
from crispasr_amd import ggml
from gpu_util import assert_parity, upload
from test_fattn_pipe_ends_gpu import _behind
from test_relpos_gpu import make, strided

pytestmark = pytest.mark.gpu


def _between(t, n, before):
    """rows before .. before + n - 1 of a tensor; the others' bits are NaN's"""
    buf = t.buf.copy()
    for i2 in range(t.ne[2]):
        for i1 in [*range(before), *range(before + n, t.ne[1])]:
            at = t.offset + i1 * t.nb[1] + i2 * t.nb[2]
            buf[at:at + 2 * t.ne[0]] = 0xFF
    return dataclasses.replace(t, buf=buf, offset=t.offset + before * t.nb[1], ne=(t.ne[0], n, t.ne[2], t.ne[3]))


def _check(seed, D, Nq, Nkv, H, B, add, add_type=ora.F32, hide=None):
    print("case", D, Nq, Nkv, H, B, add, hide, flush=True)
    c = make(seed, D, Nq, Nkv, H, B, add=add, add_type=add_type, qgain=0.7)
    if hide is not None:                                     # the last sequence's keys from `hide` on, for every query
        x = np.zeros((B, 1, Nq, Nkv), np.float32)
        x[-1, :, :, hide:] = -np.inf
        c["add"] = ora.from_f32(x, add_type)
    qu = strided(np.float32(0.7) * ora.randn(seed + 10, (B, H, Nq, D)), "cont")
    k, v = (_behind(ora.from_f32(ora.randn(seed + i, (B, H, Nkv + 70, D)), ora.F16), Nkv, 70) for i in (11, 12))
    NR = Nq + Nkv - 1
    r = _between(ora.from_f32(ora.randn(seed + 13, (1, H, NR + 200, D)), ora.F16), NR, 100)
    ref = ora.flash_attn_ext(qu, k, v, ora.relpos_bias(c["qv"], r, c["add"], c["scale"], Nkv), c["scale"])
    assert np.isfinite(ref).all()
    da = upload(c["add"]) if c["add"] is not None else None
    got = ggml.flash_attn_relpos(upload(qu), upload(c["qv"]), upload(k), upload(v), upload(r), da, c["scale"]).numpy_f32()
    assert_parity(got, ref, max_abs_tol=5e-3)                # (as in test_fattn_relpos_grid_gpu)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("add,add_type", [(None, ora.F32), ("perhead", ora.F32), ("padlong", ora.F16)])
@pytest.mark.parametrize("Nq,Nkv", [(1, 1), (5, 20), (20, 20), (32, 32), (40, 31), (33, 33), (64, 64), (50, 65), (97, 96), (130, 97), (100, 200)])
def test_rows_behind_the_ends(D, add, add_type, Nq, Nkv):
    _check(7400 + Nq + Nkv, D, Nq, Nkv, 2, 3 if add == "padlong" else 1, add, add_type)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,hide", [(20, 7), (20, 0), (32, 1), (50, 32), (50, 31), (50, 0), (64, 33), (96, 64), (96, 30), (130, 96), (200, 0)])
def test_hidden_ends(D, T, hide):
    _check(7500 + T + hide, D, T, T, 2, 2, None, hide=hide)
