"""The tile kernel under masks that hide the end of the key range (tiles it does not walk) and its orders of workgroups:
ends at every place of a tile, rows and waves that differ, queries that see nothing, hidden keys that hold NaN bits, grids of
less than one, one and several workgroups per CU and of sizes the ordering rule leaves alone."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def masked_case(visible, seed, **kw):
    """visible: bool [Bm, Hm, Nq, Nkv]"""
    case = make_case(seed=seed, Nq=visible.shape[2], Nkv=visible.shape[3], **kw)
    case["mask"] = ora.from_f32(np.where(visible, 0.0, -np.inf).astype(np.float32), ora.F16)
    return case


def ends(Nq, Nkv):
    j, i = np.arange(Nkv)[None, :], np.arange(Nq)[:, None]
    yield "causal", j <= i + Nkv - Nq
    yield "causal from zero", j <= i
    yield "one length", (j < 385) & (i >= 0)
    yield "lengths by row", j < (i * 131) % Nkv
    yield "first rows see most", j < Nkv - 2 * i
    yield "one row sees the last key", (j < 64) | ((i == Nq // 2) & (j == Nkv - 1))
    yield "late holes", (j < 70) | ((j == 511) & (i % 50 == 3))
    yield "nothing", np.zeros((Nq, Nkv), bool)


# (head size, tile_variant: query blocks per wave + 16 * key split); 80 runs on rows zero-padded to 128
FORMS = [(128, 0x11), (80, 0x11), (64, 0x12), (64, 0x11), (128, 0x21), (64, 0x21)]


@pytest.mark.parametrize("D,variant", FORMS)
@pytest.mark.parametrize("Nq,Nkv,softcap", [(150, 640, 0.0), (257, 577, 0.0), (40, 519, 0.0), (129, 1026, 0.0), (130, 530, 20.0)])
def test_hidden_ends(D, variant, Nq, Nkv, softcap):
    if softcap and variant == 0x21:
        pytest.skip("the key-split form has no soft cap")
    for name, visible in ends(Nq, Nkv):
        print("case", D, hex(variant), Nq, Nkv, name, flush=True)
        case = masked_case(visible[None, None], 5000 + Nkv, D=D, Hq=4, Hkv=2)
        case["softcap"] = softcap
        ref = run_oracle(case)
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), ref, name)
        if not softcap and Nkv > 1000:
            assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=2), ref, name + ", two ranges")


@pytest.mark.parametrize("D,variant", [(128, 0x11), (64, 0x12), (64, 0x21)])
@pytest.mark.parametrize("Hq,Hkv,B,Hm,Bm", [(8, 2, 8, 1, 8), (16, 16, 8, 1, 1), (4, 4, 5, 4, 5), (3, 1, 2, 1, 2), (24, 8, 5, 1, 5)])
def test_orders_of_workgroups(D, variant, Hq, Hkv, B, Hm, Bm):
    """every (query tile, head, sequence) once, with its own mask: 2 to 5 query tiles x 6 to 128 heads"""
    Nq, Nkv = 260, 514
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    visible = np.empty((Bm, Hm, Nq, Nkv), bool)
    for b in range(Bm):
        for h in range(Hm):
            visible[b, h] = (j < 30 + 61 * b + 17 * h) | (j < i // 4)
    print("case", D, hex(variant), Hq, B, Hm, Bm, flush=True)
    case = masked_case(visible, 5100 + Hq, D=D, Hq=Hq, Hkv=Hkv, B=B)
    case["max_bias"] = 8.0 if Hm > 1 else 0.0
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), run_oracle(case))


@pytest.mark.parametrize("D,variant", [(128, 0x11), (64, 0x12)])
def test_hidden_nan_rows(D, variant):
    """slots behind the end were never written: NaN bits in them must not show"""
    visible = np.broadcast_to(np.arange(704)[None, :] < 301, (140, 704))
    case = masked_case(visible[None, None], 5200, D=D, Hq=4, Hkv=2)
    ref = run_oracle(case)
    for t in (case["k"], case["v"]):
        t.buf[t.offset:].reshape(2, 704, -1)[:, 301:] = 0xFF
    print("case", D, hex(variant), flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), ref)
