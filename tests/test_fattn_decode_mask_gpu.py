"""The decode kernel under masks that hide whole 32-key steps: hidden ends, beginnings and holes, rows that differ, single
visible keys around the edges of steps, 512-key windows and splits, and hidden keys that hold NaN bits (never read)."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def masked_case(visible, seed, D, Hq, Hkv, ktype, max_bias=0.0, **kw):
    """visible: bool [Bm, Hm, Nq, Nkv]"""
    Bm, Hm, Nq, Nkv = visible.shape
    case = make_case(seed=seed, D=D, Nq=Nq, Nkv=Nkv, Hq=Hq, Hkv=Hkv, B=max(Bm, kw.pop("B", 1)), ktype=ktype, **kw)
    case["mask"] = ora.from_f32(np.where(visible, 0.0, -np.inf).astype(np.float32), ora.F16)
    case["max_bias"] = max_bias
    return case


def patterns(Nq, Nkv):
    j, i = np.arange(Nkv)[None, :], np.arange(Nq)[:, None]
    yield "prefix", j <= Nkv // 3 + i
    yield "suffix", j >= Nkv - 1 - i
    yield "edges", (j % 512 == 511) | (j % 512 == 32) | (j == Nkv - 1)
    yield "holes", ((j // 32 + i) % 5 == 0) & (j % 32 < 7)
    yield "one row sees nothing", (i > 0) & (j % 96 < 33)
    yield "nothing", np.zeros((Nq, Nkv), bool)


FORMS = [(64, ora.F16), (128, ora.F16), (80, ora.F16), (64, ora.Q8_0), (128, ora.Q8_0), (128, ora.Q4_0), (64, ora.Q5_1)]


@pytest.mark.parametrize("D,ktype", FORMS)
@pytest.mark.parametrize("Nq,Hq,Hkv,Nkv,n_splits", [(1, 8, 2, 8, 1), (1, 8, 2, 547, 1), (1, 4, 4, 2049, 1), (1, 8, 2, 2048, 3), (5, 4, 4, 1500, 4),
                                                    (3, 8, 2, 1031, 0), (13, 2, 2, 700, 2), (20, 4, 2, 520, 1)])
def test_hidden_steps(D, ktype, Nq, Hq, Hkv, Nkv, n_splits):
    for name, visible in patterns(Nq, Nkv):
        print("case", D, ktype, Nq, Nkv, name, flush=True)
        case = masked_case(visible[None, None], 4000 + Nkv, D, Hq, Hkv, ktype)
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=n_splits), run_oracle(case), name)


@pytest.mark.parametrize("D,ktype", [(64, ora.F16), (128, ora.Q8_0)])
@pytest.mark.parametrize("n_splits", [0, 1, 5])
def test_masks_per_head_and_sequence(D, ktype, n_splits):
    rng = np.random.default_rng(5)
    visible = np.zeros((3, 4, 2, 903), bool)
    for b in range(3):
        for h in range(4):
            lo, n = rng.integers(0, 900), rng.integers(1, 400)
            visible[b, h, :, lo:lo + n] = True
    print("case", D, ktype, n_splits, flush=True)
    case = masked_case(visible, 4100, D, 8, 2, ktype, max_bias=8.0)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=n_splits), run_oracle(case))


@pytest.mark.parametrize("D,ktype", [(64, ora.F16), (128, ora.F16), (128, ora.Q8_0)])
def test_hidden_nan_rows(D, ktype):
    """slots behind the rows so far were never written: NaN bits there must not show, at the end of the last visible step either"""
    visible = np.broadcast_to(np.arange(640)[None, :] < 301, (1, 640))
    case = masked_case(visible[None, None], 4200, D, 8, 2, ktype)
    ref = run_oracle(case)
    for t in (case["k"], case["v"]):
        rows = t.buf[t.offset:].reshape(2, 640, -1)
        rows[:, 301:] = 0xFF if ktype == ora.F16 else np.tile(np.r_[0xFF, 0xFF, np.full(32, 0x11)].astype(np.uint8), D // 32)
    print("case", D, ktype, flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA), ref)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=1), ref)


# the look at the mask: from five steps a split on, up to 128 for one row (two requests from 65 on) and 16 for 2 .. 8 rows
LIMITS = [(1, 128), (1, 129), (1, 2048), (1, 2049), (1, 4096), (1, 4097), (2, 161), (4, 512), (5, 512), (8, 507), (9, 512), (8, 513)]


@pytest.mark.parametrize("D,ktype", [(64, ora.F16), (128, ora.Q8_0), (64, ora.Q5_1)])
@pytest.mark.parametrize("Nq,Nkv", LIMITS)
def test_looks_at_their_limits(D, ktype, Nq, Nkv):
    """one visible key, or none, for each row: the first and the last of a wave's steps, of a request and of the split"""
    keys = sorted({0, 31, 32, 127, 128, 159, 160, 511, 512, 2047, 2048, 2175, Nkv - 33, Nkv - 8, Nkv - 1})
    keys = [k for k in keys if 0 <= k < Nkv]
    visible = np.zeros((len(keys), 1, Nq, Nkv), bool)                    # a sequence for each key, rows from the last one up
    for b, k in enumerate(keys):
        for i in range(Nq):
            visible[b, 0, Nq - 1 - i, max(k - 37 * i, 0)] = i == 0 or (b + i) % 3 != 0
    print("case", D, ktype, Nq, Nkv, flush=True)
    case = masked_case(visible, 4300 + Nkv + Nq, D, 2, 2, ktype)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=1), run_oracle(case))
