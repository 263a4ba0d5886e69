"""Decode calls on a caller's workspace that holds fewer key ranges than the call is cut into on its own: workspaces that were sized when
calls were cut into fewer."""
import pytest
import torch

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_oracle, upload
from test_decode_ranges import _was_cut

pytestmark = pytest.mark.gpu

# (type, head size, query heads, KV heads, sequences, rows, keys) whose ranges were fewer
CALLS = [("f16", 64, 20, 20, 8, 1, 4096), ("q8_0", 64, 20, 20, 8, 1, 1168), ("f16", 64, 20, 20, 1, 5, 560)]
TYPES = {"f16": ora.F16, "q8_0": ora.Q8_0}


def _bytes(n):
    return torch.empty(n, dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("call", CALLS, ids=str)
def test_ranges_that_fit(call):
    kt, D, hq, hkv, B, nq, nkv = call
    case = make_case(seed=920, D=D, Nq=nq, Nkv=nkv, Hq=hq, Hkv=hkv, B=B, ktype=TYPES[kt])
    q, k, v = (upload(case[t]) for t in "qkv")
    ref, before, part = run_oracle(case), _was_cut(*call), hq * B * nq * (D + 2) * 4
    need = ggml.flash_attn_workspace_size(q, k, v, None, case["scale"])
    assert need > before * part
    print("case", call, before, need // part, flush=True)
    for room in (before * part, (need // part - 1) * part, need):
        ws = _bytes(room + 4096)
        ws[room:] = 0xA5
        assert_parity(ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=ws[:room]).numpy_f32(), ref, "%s in %d bytes" % (call, room))
        assert (ws[room:] == 0xA5).all()
    with pytest.raises(ggml.Mi355xError, match="workspace"):
        ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=_bytes(before * part - 16))


def test_behind_rounded_queries_and_a_position_mask():
    """the same where the attention call has the rest of a larger workspace: q_quant, and relative positions with the kernel named"""
    call = CALLS[1]
    kt, D, hq, hkv, B, nq, nkv = call
    case = make_case(seed=921, D=D, Nq=nq, Nkv=nkv, Hq=hq, Hkv=hkv, B=B, ktype=TYPES[kt])
    q, k, v = (upload(case[t]) for t in "qkv")
    before, part = _was_cut(*call), hq * B * nq * (D + 2) * 4
    inner = ggml.flash_attn_workspace_size(q, k, v, None, case["scale"])
    whole = ggml.flash_attn_workspace_size(q, k, v, None, case["scale"], q_quant=ggml.Q8_0)
    small = whole - inner + before * part
    want = ggml.flash_attn_ext(q, k, v, None, case["scale"], q_quant=ggml.Q8_0).numpy_f32()
    assert_parity(ggml.flash_attn_ext(q, k, v, None, case["scale"], q_quant=ggml.Q8_0, workspace=_bytes(small)).numpy_f32(), want, "q_quant")
    with pytest.raises(ggml.Mi355xError, match="workspace"):
        ggml.flash_attn_ext(q, k, v, None, case["scale"], q_quant=ggml.Q8_0, workspace=_bytes(small - 16))

    D, H, nq, nkv = 64, 20, 5, 560
    qu, qv, k, v = (upload(ora.from_f32(ora.randn(930 + i, (1, H, n, D)), t)) for i, (n, t) in enumerate(((nq, ora.F32), (nq, ora.F32), (nkv, ora.F16), (nkv, ora.F16))))
    r = upload(ora.from_f32(ora.randn(935, (1, H, nq + nkv - 1, D)), ora.F16))
    kw = dict(kernel=ggml.KERNEL_DECODE_MMA)
    whole = ggml.flash_attn_relpos_workspace_size(qu, qv, k, v, r, None, 0.1, **kw)
    m = ggml.Tensor(None, ggml.F16, (nkv, nq, H, 1))
    inner = ggml.flash_attn_workspace_size(qu, k, v, m, 0.1, **kw)
    before, part = _was_cut("f16", D, H, H, 1, nq, nkv), H * nq * (D + 2) * 4
    assert inner > before * part
    small = whole - inner + before * part
    want = ggml.flash_attn_relpos(qu, qv, k, v, r, None, 0.1, **kw).numpy_f32()
    print("case relative positions", whole, small, flush=True)
    assert_parity(ggml.flash_attn_relpos(qu, qv, k, v, r, None, 0.1, workspace=_bytes(small), **kw).numpy_f32(), want, "relative positions")
    with pytest.raises(ggml.Mi355xError, match="workspace"):
        ggml.flash_attn_relpos(qu, qv, k, v, r, None, 0.1, workspace=_bytes(small - 16), **kw)
