"""Which kernel runs a tile kernel's call, and with how many waves a workgroup, planned without a GPU."""
import pytest

import crispasr_amd as ca
from crispasr_amd import ggml


def _t(type_, ne):
    return ca.Tensor(None, type_, ne)


def _form(D, Nq, Nkv, H, B=1, ktype=ggml.F16, mask=None, **kw):
    q, k = _t(ggml.F32, (D, Nq, H, B)), _t(ktype, (D, Nkv, H, B))
    kw.setdefault("kernel", ggml.KERNEL_MMA)
    return tuple(ggml.flash_attn_plan_form(q, k, k, _t(ggml.F16, (Nkv, Nq, mask, 1)) if mask else None, 0.1, **kw).values())


@pytest.mark.parametrize("D,Nq,B", [(64, 1500, 4), (64, 1000, 4), (128, 750, 4)])
def test_eight_waves_where_they_fill_the_cus_as_evenly(D, Nq, B):
    assert _form(D, Nq, Nq, 20, B) == (1, 8)
    assert _form(D, Nq, Nq, 20, B, tile_variant=0x12 if D == 64 else 0x11) == (1, 4)      # (a form by name has four)
    assert _form(D, Nq, Nq, 20, B, logit_softcap=30.0) == (0, 4)
    assert _form(D, Nq, Nq, 10, 1) in ((1, 4), (0, 4))


def test_masked_calls():
    for Nkv, variant, pipelined in ((384, 0x11, 1), (383, 0x11, 0), (382, 0x11, 0), (384, 0x21, 1), (385, 0x21, 1), (385, 0x11, 0), (383, 0x21, 0)):
        assert _form(128, 200, Nkv, 8, mask=1, tile_variant=variant) == (pipelined, 4), (Nkv, variant)
    assert _form(128, 200, 1024, 8, mask=1, tile_variant=0x21, n_splits=2) == (1, 4)
    assert _form(128, 200, 1024, 8, mask=1, tile_variant=0x21, n_splits=4) == (0, 4)       # (ranges of 256 keys)
    assert _form(128, 200, 1024, 8, mask=1, max_bias=8.0) == (0, 4)
    assert _form(64, 1500, 1500, 20, 4, mask=1) == (0, 4)
    assert _form(64, 200, 1024, 8, ktype=ggml.F32) == (1, 4)                               # (on f16 copies)
    assert _form(128, 1, 1024, 8, kernel=ggml.KERNEL_AUTO) == (0, 0)


@pytest.mark.parametrize("mask", [None, 1])
def test_ranges_longer_than_request_addresses(mask):
    """1000 rows 2 MiB apart lie beyond 2^31 bytes: the tile kernel's, with 64-bit addresses"""
    def pipelined(pitch, ns=1):
        q, k = _t(ggml.F32, (128, 100, 4, 1)), ca.Tensor(None, ggml.F16, (128, 1000, 4, 1), (2, pitch, 256, pitch * 1000))
        return ggml.flash_attn_plan_form(q, k, k, _t(ggml.F16, (1000, 100, mask, 1)) if mask else None, 0.1, kernel=ggml.KERNEL_MMA, tile_variant=0x11, n_splits=ns)["pipelined"]
    assert pipelined(1 << 20) == 1 and pipelined(1 << 21) == 0 and (mask or pipelined(1 << 21, 3) == 1)


# (256 CUs: 224 workgroups of 64 queries leave an eighth of them without one)
@pytest.mark.parametrize("Nq,H,B,least", [(1, 1, 1, 768), (1500, 8, 1, 768), (1792, 8, 1, 768), (128, 7, 16, 768), (1856, 8, 1, 1152), (2048, 8, 1, 1152), (2049, 8, 1, None)])
def test_waves_of_different_keys(Nq, H, B, least):
    def form(Nkv, D=64, mask=None, kernel=ggml.KERNEL_MMA, **kw):
        q, k = _t(ggml.F32, (D, Nq, H, B)), _t(ggml.F16, (D, Nkv, H, B))
        return ggml.flash_attn_plan_kernel_form(q, k, k, _t(ggml.F16, (Nkv, Nq, 1, 1)) if mask else None, 0.1, kernel=kernel, **{"n_splits": 1, **kw})
    for Nkv in (100, 767, 768, 1151, 1152, 4000):
        assert form(Nkv) == (ggml.FORM_KEYS_APART if least and Nkv >= least else ggml.FORM_GENERAL), Nkv
    for other in (dict(D=128), dict(D=56), dict(mask=1), dict(tile_variant=0x21), dict(logit_softcap=20.0), dict(kernel=ggml.KERNEL_VEC)):
        assert form(1200, **other) != ggml.FORM_KEYS_APART, other
    if least == 768:
        assert form(1536, n_splits=2) == (ggml.FORM_KEYS_APART if H * B * ((Nq + 63) // 64) * 2 <= 224 else ggml.FORM_GENERAL)
        assert form(1408, n_splits=2) == ggml.FORM_GENERAL                                 # (ranges of 704 keys)


# (more than a quarter of the CUs, at most half of them, with workgroups of 128 queries)
@pytest.mark.parametrize("Nq,H,Nkv,mask,split", [(48, 100, 64, None, 2), (49, 100, 32, None, 1), (64, 100, 33, None, 1), (65, 100, 32, None, 2), (100, 100, 33, None, 1), (100, 100, 65, None, 2),
                                                 (64, 100, 17, 1, 1), (64, 100, 64, 1, 1), (65, 100, 17, 1, 2), (1185, 12, 33, 1, 2), (1185, 12, 64, 1, 2), (100, 64, 64, None, 2), (100, 129, 32, 1, 1)])
def test_pairs_of_a_tile_of_keys(Nq, H, Nkv, mask, split):
    q, k = _t(ggml.F32, (128, Nq, H, 1)), _t(ggml.F16, (128, Nkv, H, 1))
    assert ggml.flash_attn_plan_details(q, k, k, _t(ggml.F16, (Nkv, Nq, mask, 1)) if mask else None, 0.1, kernel=ggml.KERNEL_MMA)["key_split"] == split
