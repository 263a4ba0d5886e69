"""The pipelined tile kernel (fattn_pipe.hip) at the edges of its blocks: 32-key blocks, odd and even numbers of steps, one
step only, rings that wrap, query tails, each form by name, references that have to climb during the key loop."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

# (head size, tile_variant: query blocks per wave + 16 * key split); 48 and 80 run on rows zero-padded to 64 and 128
FORMS = [(64, 0x12), (64, 0x11), (64, 0x21), (128, 0x11), (48, 0x11), (48, 0x21), (80, 0x11)]


@pytest.mark.parametrize("D,variant", FORMS)
@pytest.mark.parametrize("Nq,Nkv", [(1, 1), (33, 31), (64, 32), (65, 33), (128, 63), (129, 64), (255, 65), (257, 96), (96, 127), (160, 128),
                                    (31, 129), (130, 257), (200, 260), (70, 511)])
def test_edges_of_blocks_and_steps(D, variant, Nq, Nkv):
    case = make_case(seed=3000 + Nq + Nkv, D=D, Nq=Nq, Nkv=Nkv, Hq=4, Hkv=2, B=2, kv_layout="thd" if Nkv % 2 else "gap")
    print("case", D, hex(variant), Nq, Nkv, flush=True)
    ref = run_oracle(case)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), ref)
    if Nkv > 128:
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=3), ref)


@pytest.mark.parametrize("D,variant", FORMS)
@pytest.mark.parametrize("Nkv,climb", [(96, 40.0), (230, 90.0), (333, 12.0)])
def test_scores_that_climb(D, variant, Nkv, climb):
    """every few blocks a row's scores leave the range of the reference taken so far; every third row falls instead"""
    case = make_case(seed=3100 + Nkv, D=D, Nq=70, Nkv=Nkv, Hq=2, B=2)
    q, k = to_f32(case["q"]), to_f32(case["k"])
    k[..., 0] = np.sqrt(np.linspace(0.0, 1.0, Nkv, dtype=np.float32)) * 4.0
    q[..., 0] = climb / 4.0 / case["scale"]
    q[:, :, ::3, 0] *= -1.0
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, ora.F16)
    print("case", D, hex(variant), Nkv, climb, flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), run_oracle(case))
