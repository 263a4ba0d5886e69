"""Vector copies on both sides of the line from which their arguments' head is in registers (64 Ki units of 16 stored bytes): every type,
one to four walked dimensions, rows with gaps, against torch's own conversion, bytes around the destination included."""
import pytest
import torch

import crispasr_amd as ca
from crispasr_amd import ggml

pytestmark = pytest.mark.gpu

TYPES = {"f32": (ggml.F32, torch.float32, 4), "f16": (ggml.F16, torch.float16, 2)}


@pytest.mark.parametrize("src,dst", [("f32", "f16"), ("f16", "f32"), ("f32", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("ne,gap", [((16, 32768), 0), ((16, 32769), 0), ((64, 8191, 3), 8), ((24, 37, 41, 19), 16), ((8, 7, 9361), 24), ((1000, 263, 2, 2), 0)])
def test_copies(src, dst, ne, gap):
    st, sd, sb = TYPES[src]
    dt, dd, db = TYPES[dst]
    ne = ne + (1,) * (4 - len(ne))
    print("case", src, dst, ne, gap, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(ne[1])
    x = torch.randn(ne[3], ne[2], ne[1], ne[0] + gap, device="cuda", generator=g).to(sd)
    # token-major destination rows between guard values: [ne3][ne1][ne2][ne0 + gap]
    n = ne[3] * ne[1] * ne[2] * (ne[0] + gap)
    out = torch.full((n + 64,), 7.0, device="cuda", dtype=dd)
    row, drow = (ne[0] + gap) * sb, (ne[0] + gap) * db
    s = ca.Tensor(x.view(torch.uint8).reshape(-1), st, ne, (sb, row, row * ne[1], row * ne[1] * ne[2]))
    d = ca.Tensor(out.view(torch.uint8), dt, ne, (db, drow * ne[2], drow, drow * ne[1] * ne[2]), 32 * db)
    ca.cpy(s, d)
    want = torch.full_like(out, 7.0)
    want[32:32 + n].view(ne[3], ne[1], ne[2], ne[0] + gap)[..., :ne[0]] = x[..., :ne[0]].permute(0, 2, 1, 3).to(dd)
    assert torch.equal(out.view(torch.uint8), want.view(torch.uint8))
