"""The fused rel-pos attention kernel at the edges of its tiles, table blocks and workgroup widths: 2 to 4 waves, one to many
steps, lengths that end inside and between tiles, grids below, at and above one workgroup per CU."""
import numpy as np
import pytest

import oracle as ora
from crispasr_amd import ggml
from gpu_util import assert_parity, upload
from test_relpos_gpu import make, strided

pytestmark = pytest.mark.gpu


def check(seed, D, Nq, Nkv, H, B, add, add_type=ora.F32, layout="thd"):
    print("case", D, Nq, Nkv, H, B, add, flush=True)
    c = make(seed, D, Nq, Nkv, H, B, add=add, add_type=add_type, layout=layout, qgain=0.7)
    qu = strided(np.float32(0.7) * ora.randn(seed + 10, (B, H, Nq, D)), layout)
    k, v = (ora.from_f32(ora.randn(seed + i, (B, H, Nkv, D)), ora.F16) for i in (11, 12))
    ref = ora.flash_attn_ext(qu, k, v, ora.relpos_bias(c["qv"], c["r"], c["add"], c["scale"], Nkv), c["scale"])
    da = upload(c["add"]) if c["add"] is not None else None
    got = ggml.flash_attn_relpos(upload(qu), upload(c["qv"]), upload(k), upload(v), upload(c["r"]), da, c["scale"]).numpy_f32()
    # Both sides round mask values to f16 from sums that differ by what f16 operands leave (1e-3): a value in [4, 8) can land
    # 2^-8 apart.  Its probability then changes by at most p (1 - p) 2^-8 <= 1e-3, the result by that times |v - result|, up
    # to 5 among millions of normal values.  The 2-norm keeps the ordinary bound.
    assert_parity(got, ref, max_abs_tol=5e-3)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("add,add_type", [(None, ora.F32), ("padlong", ora.F32), ("padlong", ora.F16), ("perhead", ora.F32)])
@pytest.mark.parametrize("Nq,Nkv", [(1, 33), (32, 32), (64, 95), (65, 64), (96, 96), (97, 129), (128, 63), (129, 160), (193, 225), (31, 300)])
def test_edges_of_tiles_and_widths(D, add, add_type, Nq, Nkv):
    check(6000 + Nq + Nkv, D, Nq, Nkv, 2, 5 if add == "padlong" else 1, add, add_type)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,H,B", [(150, 8, 16), (390, 8, 8), (200, 8, 24), (260, 4, 50)])
def test_grids(D, T, H, B):
    check(6100 + T, D, T, T, H, B, "padlong")


# 64-wide heads: calls that run with 2, 3 and 4 waves a workgroup, one and several workgroups on a CU
@pytest.mark.parametrize("add,add_type", [(None, ora.F32), ("padlong", ora.F32), ("padlong", ora.F16)])
@pytest.mark.parametrize("T,H,B", [(100, 4, 4), (129, 8, 16), (200, 8, 24), (70, 8, 20), (97, 8, 22), (128, 8, 20), (121, 8, 40)])
def test_widths_by_grid(T, H, B, add, add_type):
    check(6200 + T, 64, T, T, H, B, add, add_type)
