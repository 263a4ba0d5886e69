"""Vector copies into destinations that are whole 128-byte lines, whole 32-byte sectors, or neither: the stores of each are the kernel's
own choice of cache bits, the bytes are the oracle's, and rows between lines cost no more than the bytes they have."""
import numpy as np
import pytest
import torch

import crispasr_amd as ca
import oracle as ora
from cases import to_f32
from crispasr_amd import ggml
from gpu_util import upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stype,dtype", [(ora.F32, ora.F16), (ora.F16, ora.F16), (ora.F32, ora.F32), (ora.F16, ora.F32), (ora.Q8_0, ora.F32), (ora.Q5_1, ora.F32)])
@pytest.mark.parametrize("ne0,gap,lead", [(64, 0, 0), (64, 0, 16), (64, 0, 32), (64, 32, 0), (64, 16, 0), (96, 0, 0), (32, 128, 128), (160, 48, 64)])
def test_destinations(stype, dtype, ne0, gap, lead):
    """gap and lead in bytes: between the heads' rows, ahead of the first"""
    T, H = 37, 5
    src = ora.from_f32(ora.randn(940 + ne0 + gap, (1, H, T, ne0)), stype)
    es, pitch = ora.TYPE_SIZE[dtype], ora.row_size(dtype, ne0) + gap
    raw = np.full(lead + pitch * H * T + 64, 0xA5, np.uint8)
    view = (dtype, (ne0, T, H, 1), (es, pitch * H, pitch, pitch * H * T), lead)
    want = ora.Tensor(raw.copy(), *view)
    values = to_f32(src).reshape(H, T, ne0)
    cast = values.astype(np.float16) if dtype == ora.F16 else values.astype(np.float32)
    for h in range(H):
        for t in range(T):
            at = lead + pitch * (t * H + h)
            want.buf[at:at + ne0 * es] = cast[h, t].view(np.uint8)
    print("copy", stype, dtype, ne0, gap, lead, flush=True)
    got = ca.Tensor.from_host(raw, *view)
    ca.cpy(upload(src), got)
    assert np.array_equal(got.to_host(), want.buf)


def _us(src, dst):
    best = 1e30
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(20):
            ca.cpy(src, dst)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 50.0)
    return best


def test_rows_between_lines_cost_their_bytes():
    """64 heads x 2048 Q8_0 rows of 128 read back as F32, token by token, heads 512 bytes apart and 544: 6% more memory under the same bytes,
    and a row touches five lines where it filled four - a quarter more.  Lines that are not whole, marked non-temporal, cost 1.7 times."""
    T, H = 2048, 64
    src = ggml.Tensor.empty(ggml.Q8_0, (128, T, H))
    src.buf.zero_()
    us = []
    for pitch in (512, 544):
        buf = torch.zeros(pitch * H * T, dtype=torch.uint8, device="cuda")
        us.append(_us(src, ca.Tensor(buf, ggml.F32, (128, T, H), (4, pitch * H, pitch, pitch * H * T))))
    print("rows of 512 bytes at 512 and at 544: %.1f, %.1f us" % tuple(us), flush=True)
    assert us[1] < 1.4 * us[0], us
