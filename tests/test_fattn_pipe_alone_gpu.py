"""The pipelined tile kernel's form whose waves take different keys of the same 64 queries (64-wide heads, a workgroup a CU at most, 768 keys
of a range and more): block and step counts of every remainder, waves without a block of their own in the last step, query tails,
ranges, references that climb, NaN bits behind the last key."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, kernel_form, run_gpu, run_oracle
from test_fattn_pipe_ends_gpu import _behind

pytestmark = pytest.mark.gpu


def _check(case, ns=1):
    assert kernel_form(case, kernel=ggml.KERNEL_MMA, n_splits=ns) == ggml.FORM_KEYS_APART
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, n_splits=ns), run_oracle(case))


@pytest.mark.parametrize("Nq,Nkv", [(40, 768), (64, 799), (1, 896), (16, 897), (63, 927), (64, 928), (65, 929), (100, 959), (127, 960), (128, 961), (129, 991), (31, 992), (70, 993),
                                    (33, 1023), (96, 1024), (97, 1025), (200, 1151), (30, 1500), (65, 1536)])
def test_remainders(Nq, Nkv):
    case = make_case(seed=5200 + Nkv, D=64, Nq=Nq, Nkv=Nkv, Hq=4, Hkv=2, B=2, q_layout="thd", kv_layout="thd" if Nkv % 2 else "gap")
    print("case", Nq, Nkv, flush=True)
    _check(case)


@pytest.mark.parametrize("ns,Nkv", [(2, 1536), (2, 1600), (2, 1920), (3, 2700), (3, 2753)])
def test_ranges(ns, Nkv):
    case = make_case(seed=5300 + Nkv, D=64, Nq=70, Nkv=Nkv, Hq=4, Hkv=2)
    print("case", ns, Nkv, flush=True)
    _check(case, ns)


@pytest.mark.parametrize("Nkv,climb", [(900, 40.0), (1000, 90.0), (1100, 12.0)])
def test_scores_that_climb(Nkv, climb):
    case = make_case(seed=5400 + Nkv, D=64, Nq=70, Nkv=Nkv, Hq=2, B=2)
    q, k = to_f32(case["q"]), to_f32(case["k"])
    k[..., 0] = np.sqrt(np.linspace(0.0, 1.0, Nkv, dtype=np.float32)) * 4.0
    q[..., 0] = climb / 4.0 / case["scale"]
    q[:, :, ::3, 0] *= -1.0
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, ora.F16)
    print("case", Nkv, climb, flush=True)
    _check(case)


@pytest.mark.parametrize("Nkv", [896, 930, 1000, 1055])
def test_nan_bits_behind_the_last_key(Nkv):
    case = make_case(seed=5500 + Nkv, D=64, Nq=90, Nkv=Nkv + 600, Hq=4, Hkv=2, kv_layout="thd" if Nkv % 4 else "contig")
    case["k"], case["v"] = _behind(case["k"], Nkv, 600), _behind(case["v"], Nkv, 600)
    print("case", Nkv, flush=True)
    _check(case)
