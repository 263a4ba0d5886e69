"""The pipelined tile kernel's workgroups of eight waves, which it takes where they fill the CUs as evenly as twice as many of four
(more than one of those a CU): edges of blocks, steps and rings, query tails, references that climb."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, plan_details, run_gpu, run_oracle, upload

pytestmark = pytest.mark.gpu

# 26 x 5 heads: 260 workgroups of four waves, 130 of eight
FORMS = {64: dict(Nq=500, queries=256), 128: dict(Nq=250, queries=128), 96: dict(Nq=141, queries=128)}


def _form(case, **kw):
    return ggml.flash_attn_plan_form(upload(case["q"]), upload(case["k"]), upload(case["v"]), None, case["scale"], kernel=ggml.KERNEL_MMA, **kw)


def _case(D, Nkv, **kw):
    case = make_case(seed=3200 + Nkv, D=D, Nq=FORMS[D]["Nq"], Nkv=Nkv, Hq=26, Hkv=13, B=5, **kw)
    plan = plan_details(case, kernel=ggml.KERNEL_MMA)
    assert plan["queries_per_workgroup"] == FORMS[D]["queries"] and plan["n_splits"] == 1, plan
    assert _form(case) == {"pipelined": 1, "waves": 8}
    print("case", D, Nkv, flush=True)
    return case


@pytest.mark.parametrize("D", sorted(FORMS))
@pytest.mark.parametrize("Nkv", [1, 31, 32, 33, 64, 97, 128, 130, 161, 257])
def test_edges_of_blocks_and_steps(D, Nkv):
    case = _case(D, Nkv, kv_layout="thd" if Nkv % 2 else "gap")
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA), run_oracle(case))


@pytest.mark.parametrize("D", sorted(FORMS))
def test_scores_that_climb(D):
    case = _case(D, 210)
    q, k = to_f32(case["q"]), to_f32(case["k"])
    k[..., 0] = np.sqrt(np.linspace(0.0, 1.0, 210, dtype=np.float32)) * 4.0
    q[..., 0] = 90.0 / 4.0 / case["scale"]
    q[:, :, ::3, 0] *= -1.0
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, ora.F16)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA), run_oracle(case))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nkv", [333, 700])
def test_ranges(D, Nkv):
    """eight waves that leave partial results: three ranges (390 workgroups of eight, 780 of four), the last one shorter"""
    case = make_case(seed=3290, D=D, Nq=FORMS[D]["Nq"], Nkv=Nkv, Hq=26, Hkv=13, B=5)
    assert _form(case, n_splits=3) == {"pipelined": 1, "waves": 8}
    print("case", D, Nkv, "in three ranges", flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, n_splits=3), run_oracle(case))
