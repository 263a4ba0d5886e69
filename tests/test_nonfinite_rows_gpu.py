"""Query rows of NaN, infinities and large values among ordinary ones: every other row is what it is without them, in every kernel and form."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

# (kernel, tile_variant, D, Nq, Nkv, Hq, B, mask)
FORMS = [
    (ggml.KERNEL_MMA, 0, 64, 70, 1000, 4, 1, None),          # the pipelined kernel: waves of different keys,
    (ggml.KERNEL_MMA, 0, 64, 70, 300, 4, 1, None),           # pairs,
    (ggml.KERNEL_MMA, 0x11, 64, 140, 200, 4, 1, None),       # one query block a wave,
    (ggml.KERNEL_MMA, 0x12, 64, 260, 200, 4, 1, None),       # two,
    (ggml.KERNEL_MMA, 0, 64, 260, 100, 16, 16, None),        # eight waves,
    (ggml.KERNEL_MMA, 0, 128, 70, 200, 4, 1, None),          # 128-wide pairs,
    (ggml.KERNEL_MMA, 0x11, 128, 140, 200, 4, 1, None),      # waves of their own
    (ggml.KERNEL_MMA, 0, 96, 70, 200, 4, 1, None),           # and padded heads;
    (ggml.KERNEL_MMA, 0, 128, 70, 200, 4, 1, "causal"),      # masked pairs
    (ggml.KERNEL_MMA, 0x11, 128, 140, 400, 4, 1, "causal"),
    (ggml.KERNEL_MMA, 0x11, 64, 140, 400, 4, 1, "causal"),   # the tile kernel
    (ggml.KERNEL_MMA, 0x21, 64, 70, 400, 4, 1, "causal"),
    (ggml.KERNEL_DECODE_MMA, 0, 64, 14, 300, 4, 1, None),
    (ggml.KERNEL_DECODE_MMA, 0, 128, 14, 300, 4, 1, None),
    (ggml.KERNEL_VEC, 0, 64, 14, 300, 4, 1, None),
]


@pytest.mark.parametrize("kernel,variant,D,Nq,Nkv,Hq,B,mask", FORMS)
@pytest.mark.parametrize("what", [np.nan, np.inf, 3.0e4])
def test_rows_on_their_own(kernel, variant, D, Nq, Nkv, Hq, B, mask, what):
    case = make_case(seed=8000 + D + Nq + Nkv, D=D, Nq=Nq, Nkv=Nkv, Hq=Hq, B=B, mask=mask)
    q = to_f32(case["q"]).copy()
    odd = np.arange(Nq) % 7 == 3                             # (rows 16 and 32 apart among them and not)
    odd[-1] = True
    q[:, :, odd, 5] = what
    case["q"] = ora.from_f32(q, ora.F32)
    print("case", kernel, hex(variant), D, Nq, Nkv, mask, what, flush=True)
    ref = run_oracle(case)                                   # [B, Nq, Hq, D]
    got = run_gpu(case, kernel=kernel, tile_variant=variant, n_splits=1)
    assert np.isfinite(ref[:, ~odd]).all()
    assert_parity(got[:, ~odd], ref[:, ~odd])
    if np.isnan(what):
        assert np.isnan(got[:, odd]).all()


@pytest.mark.parametrize("D,ktype", [(64, ora.F16), (128, ora.F16), (96, ora.F16), (64, ora.Q8_0), (128, ora.Q8_0), (128, ora.Q4_0)])
@pytest.mark.parametrize("Nq,Nkv,ns", [(1, 20, 1), (1, 33, 1), (1, 300, 1), (3, 300, 2), (1, 1500, 0), (1, 1500, 7)])
def test_decode_rows_of_nan_stay_nan(D, ktype, Nq, Nkv, ns):
    case = make_case(seed=8100 + D + Nkv, D=D, Nq=Nq, Nkv=Nkv, Hq=4, Hkv=2, ktype=ktype)
    q = to_f32(case["q"]).copy()
    q[:, 1, -1, 3] = np.nan
    case["q"] = ora.from_f32(q, ora.F32)
    print("case", D, ktype, Nq, Nkv, ns, flush=True)
    ref, got = run_oracle(case), run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=ns)
    assert np.isnan(got[:, -1, 1]).all()                     # (the exact oracle has no largest score and gives zeros; the CPU op gives NaN)
    if ktype == ora.F16:
        assert np.isnan(run_oracle(case, ora.MODE_GGML_LIKE)[:, -1, 1]).all()
    assert_parity(got[:, :, [0, 2, 3]], ref[:, :, [0, 2, 3]])
