"""Unmasked decode calls over f16 rows: one, an even and an odd number of steps a wave, ends inside a step, waves without a step, 128-wide ranges
of one step a wave and of more, padded head sizes, grids on both sides of three workgroups a CU, NaN bits behind the last key, rows too far
apart for one request's offsets; and streamed rows, whose first request takes no branch."""
import pytest
import torch

import crispasr_amd as ca
import oracle as ora
from cases import errors, make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, kernel_form, run_gpu, run_oracle
from test_fattn_pipe_ends_gpu import _behind

pytestmark = pytest.mark.gpu


def _check(case, ref, ns, what=""):
    """f16 rows: two steps under way, at (or padded to) 128 elements in ranges of one step a wave only"""
    D, Nkv = case["k"].ne[:2]
    keys = ((Nkv + ns - 1) // ns + 31) // 32 * 32
    assert kernel_form(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=ns) == (ggml.FORM_DEEP if D <= 64 or keys <= 128 else ggml.FORM_SHORT)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=ns), ref, what)


@pytest.mark.parametrize("D", [64, 128, 80, 32])
@pytest.mark.parametrize("Nkv", [1, 31, 32, 33, 96, 127, 128, 129, 160, 255, 256, 257, 289, 384, 385, 420, 512, 513, 700, 897])
def test_steps(D, Nkv):
    case = make_case(seed=7000 + D + Nkv, D=D, Nq=3, Nkv=Nkv, Hq=4, Hkv=2, kv_layout="thd" if Nkv % 2 else "gap")
    print("case", D, Nkv, flush=True)
    ref = run_oracle(case)
    for ns in (1, 3):
        _check(case, ref, ns, "%d ranges" % ns)


@pytest.mark.parametrize("D", [64, 128, 96])
@pytest.mark.parametrize("Nkv", [20, 100, 128, 150, 290, 400])
def test_nan_bits_behind_the_last_key(D, Nkv):
    case = make_case(seed=7100 + D + Nkv, D=D, Nq=1, Nkv=Nkv + 200, Hq=4, B=2, kv_layout="thd")
    case["k"], case["v"] = _behind(case["k"], Nkv, 200), _behind(case["v"], Nkv, 200)
    print("case", D, Nkv, flush=True)
    ref = run_oracle(case)
    for ns in (1, 2):
        _check(case, ref, ns, "%d ranges" % ns)


@pytest.mark.parametrize("Hq,B,deep", [(12, 64, True), (13, 64, False), (16, 64, False), (17, 64, True)])          # 768, 832, 1024 and 1088 workgroups on 256 CUs
def test_grids(Hq, B, deep):
    case = make_case(seed=7200 + Hq, D=64, Nq=1, Nkv=140, Hq=Hq, B=B)
    print("case", Hq, B, flush=True)
    assert kernel_form(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=1) == (ggml.FORM_DEEP if deep else ggml.FORM_SHORT)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=1), run_oracle(case))


@pytest.mark.parametrize("ktype", [ora.Q8_0, ora.Q4_0, ora.Q5_1])
@pytest.mark.parametrize("D", [64, 128])
def test_streamed_rows(D, ktype):
    for Nkv, ns in ((1, 1), (33, 1), (97, 1), (129, 1), (300, 2), (420, 4)):
        case = make_case(seed=7300 + D + Nkv, D=D, Nq=2, Nkv=Nkv, Hq=4, Hkv=2, ktype=ktype)
        print("case", D, ktype, Nkv, ns, flush=True)
        assert kernel_form(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=ns) == ggml.FORM_SHORT
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=ns), run_oracle(case))


def test_rows_far_apart():
    """three rows of K and V 80 MiB apart: the general form"""
    D, n, pitch = 64, 3, 80 << 20
    rows = [torch.randn(n, D, device="cuda").half() for _ in range(2)]
    far = []
    for x in rows:
        buf = torch.zeros(2 * pitch + 2 * D, dtype=torch.uint8, device="cuda")
        for i in range(n):
            buf[i * pitch:i * pitch + 2 * D] = x[i].view(torch.uint8)
        far.append(ca.Tensor(buf, ggml.F16, (D, n, 1, 1), (2, pitch, pitch * n, pitch * n)))
    q = torch.randn(D, device="cuda")
    qt = ca.Tensor(q.view(torch.uint8), ggml.F32, (D, 1, 1))
    assert ggml.flash_attn_plan_kernel_form(qt, far[0], far[1], None, 0.125, kernel=ggml.KERNEL_DECODE_MMA) == ggml.FORM_GENERAL
    out = ca.flash_attn_ext(qt, far[0], far[1], None, 0.125, kernel=ggml.KERNEL_DECODE_MMA).numpy_f32()
    k, v = (x.double().cpu() for x in rows)
    ref = (torch.softmax(0.125 * (k @ q.double().cpu()), 0) @ v).numpy()
    max_abs, rel = errors(out.reshape(-1), ref)
    assert max_abs < 2e-3 and rel < 2e-3          # (q and the probabilities are f16 in the products: 2^-11 each)
