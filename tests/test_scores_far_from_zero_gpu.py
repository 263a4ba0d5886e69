"""Scores that lie far above or below zero, all of a row's by the same amount, which the softmax does not see: the references of every kernel
and form start there."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle
from test_nonfinite_rows_gpu import FORMS

pytestmark = pytest.mark.gpu

MORE = [
    (ggml.KERNEL_DECODE_MMA, 0, 64, 1, 20, 4, 1, None),
    (ggml.KERNEL_DECODE_MMA, 0, 128, 1, 1500, 4, 1, None),
    (ggml.KERNEL_DECODE_MMA, 0, 96, 2, 700, 4, 1, None),
    (ggml.KERNEL_DECODE_MMA, 0, 128, 2, 700, 4, 1, "random_inf"),
    (ggml.KERNEL_VEC, 0, 36, 1, 375, 4, 1, None),
]


def _shifted(case, by):
    """adds `by` to every score: K's element 0 is 32, Q's such that their product is the same number in f16 and f32"""
    q, k = to_f32(case["q"]).copy(), to_f32(case["k"]).copy()
    k[..., 0] = 32.0
    factor = np.float32(case["scale"] * 1.4426950408889634)              # (the kernels' factor: they work in log2 units)
    q[..., 0] = np.float32(np.float16(by * 1.4426950408889634 / 32.0)) / factor
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, case["k"].type)
    return case


@pytest.mark.parametrize("kernel,variant,D,Nq,Nkv,Hq,B,mask", FORMS + MORE)
@pytest.mark.parametrize("by", [-900.0, -200.0, -95.0, -85.0, 95.0, 300.0])
def test_shifted_scores(kernel, variant, D, Nq, Nkv, Hq, B, mask, by):
    case = _shifted(make_case(seed=8200 + D + Nq + Nkv, D=D, Nq=Nq, Nkv=Nkv, Hq=Hq, B=B, mask=mask), by)
    print("case", kernel, hex(variant), D, Nq, Nkv, mask, by, flush=True)
    ref = run_oracle(case)
    for ns in (1, 3) if Nkv >= 300 else (1,):
        # Scores of 1300 in log2 units are sums of f32, off by up to 1e-4 each: probabilities by as much, the result by that times its spread
        assert_parity(run_gpu(case, kernel=kernel, tile_variant=variant, n_splits=ns), ref, "%d ranges" % ns)


@pytest.mark.parametrize("ktype", [ora.F32, ora.Q8_0, ora.Q4_0])
@pytest.mark.parametrize("D,Nq,Nkv", [(64, 1, 100), (64, 40, 300), (128, 1, 300), (128, 40, 300), (96, 40, 300)])
@pytest.mark.parametrize("by", [-300.0, -95.0])
def test_other_types(ktype, D, Nq, Nkv, by):
    case = _shifted(make_case(seed=8300 + D + Nq, D=D, Nq=Nq, Nkv=Nkv, Hq=4, ktype=ora.F32), by)
    if ktype != ora.F32:                             # (the blocks' other elements are zeros next to 32: scores that are all alike)
        case["k"], case["v"] = (ora.from_f32(to_f32(case[x]), ktype) for x in "kv")
    print("case", ktype, D, Nq, Nkv, by, flush=True)
    ref = run_oracle(case)
    for kernel in (ggml.KERNEL_AUTO, ggml.KERNEL_MMA) if Nq > 1 else (ggml.KERNEL_AUTO,):
        assert_parity(run_gpu(case, kernel=kernel), ref)
