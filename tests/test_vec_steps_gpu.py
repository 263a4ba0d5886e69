"""Unmasked F32 calls of few rows and keys, which the vector kernel takes before the tile kernel: on both sides of the line, and on a caller's
workspace that does not hold the vector kernel's partials."""
import pytest
import torch

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, plan_details, run_gpu, run_oracle, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,Nq,Nkv,vector", [
    (64, 20, 5, 1500, True), (64, 8, 15, 1500, True), (64, 8, 16, 1407, False), (64, 16, 32, 40, True), (64, 19, 27, 40, False),
    (128, 20, 48, 190, True), (128, 8, 16, 1500, False), (128, 25, 41, 40, False), (48, 8, 16, 1500, True), (80, 8, 16, 1400, True), (80, 8, 16, 1500, False)])
def test_both_sides_of_the_line(D, H, Nq, Nkv, vector):
    case = make_case(seed=6600 + D + Nq, D=D, Nq=Nq, Nkv=Nkv, Hq=H, ktype=ora.F32, q_layout="thd", kv_layout="thd")
    print("case", D, H, Nq, Nkv, flush=True)
    assert (plan_details(case)["kernel"] == ggml.KERNEL_VEC) == vector
    assert_parity(run_gpu(case), run_oracle(case))


@pytest.mark.parametrize("kw", [dict(Hkv=4), dict(mask="bias"), dict(softcap=20.0), dict(B=2), dict(ktype=ora.F16)])
def test_calls_next_to_the_rule(kw):
    case = make_case(seed=6700, D=64, Nq=16, Nkv=300, Hq=8, **{"ktype": ora.F32, **kw})
    assert plan_details(case)["kernel"] != ggml.KERNEL_VEC
    assert plan_details(case, n_splits=2)["kernel"] != ggml.KERNEL_VEC
    assert_parity(run_gpu(case), run_oracle(case))


def test_a_workspace_without_room_for_partials():
    """the tile kernel's, whose partials are fewer here, as before the vector kernel took such calls"""
    case = make_case(seed=6800, D=64, Nq=5, Nkv=700, Hq=12, ktype=ora.F32)
    q, k, v = (upload(case[t]) for t in "qkv")
    need = ggml.flash_attn_workspace_size(q, k, v, None, case["scale"])
    room = ggml.flash_attn_workspace_size(q, k, v, None, case["scale"], kernel=ggml.KERNEL_MMA)
    assert 0 < room < need
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")
    assert ggml.flash_attn_plan_details(q, k, v, None, case["scale"], workspace=ws)["kernel"] == ggml.KERNEL_VEC
    assert ggml.flash_attn_plan_details(q, k, v, None, case["scale"], workspace=ws[:room])["kernel"] == ggml.KERNEL_MMA
    assert_parity(ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=ws[:room]).numpy_f32(), run_oracle(case))
    assert (ws[room:] == 0xA5).all()
    with pytest.raises(ggml.Mi355xError, match="workspace"):
        ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=ws[:room - 16])


@pytest.mark.parametrize("D,Nq,Nkv,H,room", [(96, 383, 300, 1, 153600), (32, 383, 300, 1, 76800), (80, 360, 320, 1, 163840), (48, 380, 280, 1, 71680)])
def test_a_workspace_of_the_padded_copies(D, Nq, Nkv, H, room):
    """less than the vector kernel's partials take: its call in one range"""
    case = make_case(seed=6900 + D, D=D, Nq=Nq, Nkv=Nkv, Hq=H, ktype=ora.F32)
    print("case", D, Nq, Nkv, H, flush=True)
    q, k, v = (upload(case[t]) for t in "qkv")
    assert ggml.flash_attn_workspace_size(q, k, v, None, case["scale"], kernel=ggml.KERNEL_MMA) == room
    assert ggml.flash_attn_workspace_size(q, k, v, None, case["scale"]) > room
    ws = torch.full((room,), 0xA5, dtype=torch.uint8, device="cuda")
    assert_parity(ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=ws).numpy_f32(), run_oracle(case))
    with pytest.raises(ggml.Mi355xError, match="workspace"):
        ggml.flash_attn_ext(q, k, v, None, case["scale"], workspace=ws[:room - 16])
