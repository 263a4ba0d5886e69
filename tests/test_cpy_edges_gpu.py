"""The copy kernels' forms at the edges of their units: 8 elements per lane or one, quads of lanes per block, sources and
destinations that are aligned for 16-byte accesses or not, copies that reshape.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import crispasr_amd as ca
import oracle as ora
from gpu_util import upload

pytestmark = pytest.mark.gpu

TYPES = [ora.F32, ora.F16, ora.Q8_0, ora.Q4_0, ora.Q4_1, ora.Q5_0, ora.Q5_1]


def source(seed, ne0, rows, shift, step):
    """F32 rows of ne0 elements `step` floats apart from one another, `shift` floats into their buffer"""
    x = ora.randn(seed, (rows * (ne0 * step + 3) + shift,))
    x[:: 7] = -x[:: 7] * 0.0                                     # zeros of both signs
    x[3 :: 11] = x[2 :: 11][: x[3 :: 11].size]                   # ties for the largest magnitude
    return ora.Tensor(x.view(np.uint8), ora.F32, (ne0, rows, 1, 1), (4, 4 * (ne0 * step + 3 * (shift or step > 1)), 0, 0), 4 * shift)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("ne0,rows", [(32, 1), (64, 31), (32, 63), (32, 64), (96, 43), (128, 129)])
@pytest.mark.parametrize("shift", [0, 1])
def test_copies_and_set_rows_at_the_edges(dtype, ne0, rows, shift):
    src = source(900 + ne0 + rows, ne0, rows, shift, 1)
    rs = ora.row_size(dtype, ne0)
    es = ora.TYPE_SIZE[dtype]
    lead = 2 * shift if dtype != ora.F32 else 4 * shift           # a destination that starts off 16 bytes
    raw = np.full(lead + rs * rows + 32, 0xA5, np.uint8)
    nb = (es, rs, rs * rows, rs * rows)
    want = ora.Tensor(raw.copy(), dtype, (ne0, rows, 1, 1), nb, lead)
    ora.cpy_f32(src, want)
    print("copy", dtype, ne0, rows, shift, flush=True)
    got = ca.Tensor.from_host(raw, dtype, (ne0, rows, 1, 1), nb, lead)
    ca.cpy(upload(src), got)
    assert np.array_equal(got.to_host(), want.buf)
    # the same rows in another order through their indices, on a destination with its rows as they lie
    order = (np.arange(rows) * 5 + 2) % rows if rows % 5 else np.arange(rows)[::-1].copy()
    got2 = ca.Tensor.from_host(raw, dtype, (ne0, rows, 1, 1), nb, lead)
    ca.set_rows(got2, upload(src), torch.from_numpy(order.astype(np.int32)).cuda())
    w, g = want.buf[lead:lead + rs * rows].reshape(rows, rs), got2.to_host()[lead:lead + rs * rows].reshape(rows, rs)
    assert np.array_equal(g[order], w)
    # a destination of another shape with as many elements
    if rows % 2 == 0 or dtype in (ora.F32, ora.F16):
        flat = ca.Tensor.from_host(raw, dtype, (ne0 * rows,), (es, 0, 0, 0), lead)
        ca.cpy(upload(src), flat)
        assert np.array_equal(flat.to_host(), want.buf)
    # and back to F32
    if dtype != ora.F32:
        back = ca.Tensor.from_host(np.zeros(4 * ne0 * rows + 16, np.uint8), ora.F32, (ne0, rows, 1, 1), None, 4 * shift)
        ca.cpy(got, back)
        body = want.buf[lead:lead + rs * rows]
        ref = ora.fp16_to_fp32(body.view(np.uint16)) if dtype == ora.F16 else ora.dequantize(dtype, body)
        assert np.array_equal(back.to_host()[4 * shift:4 * shift + 4 * ne0 * rows].view(np.uint32), ref.reshape(-1).view(np.uint32))
