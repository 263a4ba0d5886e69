"""Unmasked calls whose rows lie further apart than the pipelined kernel's 32-bit addresses reach - a head's keys over 2 GiB and more, query
rows 32 MiB and more - are the tile kernel's, in every form a caller can name and on padded heads."""
import pytest
import torch

import crispasr_amd as ca
from cases import REL_L2_TOL
from crispasr_amd import ggml

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _rows(gen, type_, D, N, H, pitch):
    """[D, N, H] normal values in rows `pitch` bytes apart, their heads side by side; the tensor and the values"""
    dt, es = (torch.float16, 2) if type_ == ggml.F16 else (torch.float32, 4)
    x = torch.randn(N, H, D, device="cuda", generator=gen).to(dt)
    buf = torch.empty((N - 1) * pitch + es * D * H, dtype=torch.uint8, device="cuda")
    buf.view(dt).as_strided((N, H, D), (pitch // es, D, 1)).copy_(x)
    return ca.Tensor(buf, type_, (D, N, H, 1), (es, pitch, es * D, pitch * N)), x


def _check(D, Nq, Nkv, H, q_pitch, kv_pitch, variant, ns=1):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(61)
    q, qx = _rows(gen, ggml.F32, D, Nq, H, q_pitch or 4 * D * H)
    k, kx = _rows(gen, ggml.F16, D, Nkv, H, kv_pitch or 2 * D * H)
    v, vx = _rows(gen, ggml.F16, D, Nkv, H, kv_pitch or 2 * D * H)
    how = dict(kernel=ggml.KERNEL_MMA, n_splits=ns, tile_variant=variant)
    print("case", D, Nq, Nkv, H, q_pitch, kv_pitch, hex(variant), ggml.flash_attn_plan_form(q, k, v, None, D ** -0.5, **how), flush=True)
    got = ca.flash_attn_ext(q, k, v, None, D ** -0.5, **how)
    ref = torch.empty(Nq, H, D, device="cuda")
    for h in range(H):
        s = (qx[:, h] * D ** -0.5) @ kx[:, h].float().t().contiguous()
        ref[:, h] = torch.softmax(s, 1) @ vx[:, h].float()
    got = got.buf.view(torch.float32).view(Nq, H, D)
    assert float((got - ref).norm() / ref.norm()) <= REL_L2_TOL
    return ggml.flash_attn_plan_form(q, k, v, None, D ** -0.5, **how)["pipelined"]


@pytest.mark.parametrize("D,variant", [(64, 0), (64, 0x11), (64, 0x21), (64, 0x12), (128, 0), (128, 0x11), (128, 0x21)])
def test_keys_over_two_gib(D, variant):
    assert _check(D, 70, 1000, 2, 0, 2 * MIB + 256, variant) == 0
    assert _check(D, 70, 1000, 2, 0, 1 * MIB, variant) == 1


@pytest.mark.parametrize("D,variant", [(64, 0x21), (64, 0), (128, 0x21), (48, 0x21), (96, 0x21)])
def test_query_rows_far_apart(D, variant):
    _check(D, 37, 200, 1, 33 * MIB, 0, variant)


def test_a_padded_head_of_many_keys():
    """16.9 million keys of 32, one range: their copies are 2^31 bytes and more"""
    D, N = 32, (1 << 24) + 100000
    gen = torch.Generator(device="cuda")
    gen.manual_seed(62)
    q = torch.randn(16, D, device="cuda", generator=gen)
    kx = torch.randn(N, D, device="cuda", generator=gen).half()
    vx = torch.full((N, D), 0.5, device="cuda", dtype=torch.float16)
    far = torch.arange(16, device="cuda") * 7 + N - 300
    kx[far] = (q / q.norm(dim=1, keepdim=True) * 24.0).half()            # (each query's own key behind 2^31 bytes, with weight 0.1 to 1)
    vx[far] = torch.randn(16, D, device="cuda", generator=gen).half()
    s = (q.double() * D ** -0.5) @ kx.double().t().contiguous()
    ref = (torch.softmax(s, 1) @ vx.double()).float()
    del s
    t = lambda x, type_, es: ca.Tensor(x.contiguous().view(torch.uint8).view(-1), type_, (D, x.shape[0], 1, 1), (es, es * D, es * D * x.shape[0], es * D * x.shape[0]))
    qt, k, v = t(q, ggml.F32, 4), t(kx, ggml.F16, 2), t(vx, ggml.F16, 2)
    print("case", N, flush=True)
    assert ggml.flash_attn_plan_form(qt, k, v, None, D ** -0.5, kernel=ggml.KERNEL_MMA, n_splits=1)["pipelined"] == 0
    got = ca.flash_attn_ext(qt, k, v, None, D ** -0.5, kernel=ggml.KERNEL_MMA, n_splits=1).buf.view(torch.float32).view(16, D)
    # (half a million sums in a row in f32, each rounded by 2^-24 of the total: 1e-3 is four times sqrt(n) of these and f16 weights' 2^-11)
    err = float((got - ref).norm() / ref.norm())
    assert err <= 1e-3, err
