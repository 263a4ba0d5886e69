"""The native tensor views of crispasr_amd.ggml: fields, arithmetic of views, bounds and the C descriptor."""
import numpy as np
import pytest
import torch

import crispasr_amd as ca
from crispasr_amd import ggml


@pytest.mark.parametrize("type_,ne", [(ca.F32, (7,)), (ca.F16, (64, 3)), (ca.Q8_0, (64, 3, 2)), (ca.Q5_1, (32, 1, 2, 5)), (ca.F32, (0, 4, 1, 1))])
def test_fields_and_contiguous_strides(type_, ne):
    t = ca.Tensor(None, type_, ne)
    ne4 = tuple(ne) + (1,) * (4 - len(ne))
    assert (t.type, t.ne, t.nb, t.offset, t.buf) == (type_, ne4, ggml.contiguous_nb(type_, ne4), 0, None)
    blocks = ne4[0] // ggml.BLOCK_SIZE[type_]
    n = blocks * ne4[1] * ne4[2] * ne4[3]
    assert t.span() == n * ggml.TYPE_SIZE[type_]
    c = t.c()
    assert (c.type, tuple(c.ne), tuple(c.nb)) == (type_, ne4, t.nb)


def test_views_share_the_buffer_and_add_their_offsets():
    buf = torch.zeros(4096, dtype=torch.uint8)
    t = ca.Tensor(buf, ca.F16, [np.int64(64), 8], nb=(2, 128, 1024, 1024), offset=256)
    v = t.view((32, 2), (2, 128, 256, 256), 64).view((16,), (4, 64, 64, 64), offset=np.int64(8), type_=ca.F32)
    assert v.buf is buf and v.offset == 328 and v.type == ca.F32 and v.ne == (16, 1, 1, 1)
    assert v.data_ptr() == buf.data_ptr() + 328 == v.c().data and type(v) is ca.Tensor
    with pytest.raises(ggml.InvalidError, match="exceeds"):
        t.view((64, 8), t.nb, 3000).c()
    assert ca.Tensor(None, ca.F16, (8,), offset=700).c().data == 700 % 256


@pytest.mark.parametrize("bad", [torch.zeros(8), torch.zeros(2, 4, dtype=torch.uint8), torch.zeros(8, dtype=torch.uint8)[::2]])
def test_a_buffer_is_a_flat_byte_tensor(bad):
    with pytest.raises(AssertionError):
        ca.Tensor(bad, ca.F32, (1,))


def test_calls_refuse_what_is_not_a_tensor_with_memory():
    real = ca.Tensor(torch.zeros(64, dtype=torch.uint8), ca.F32, (16,))
    planned = ca.Tensor(None, ca.F32, (16,))
    with pytest.raises(AttributeError):
        ca.cpy(planned, real)
    with pytest.raises(TypeError):
        ca.cpy(real, None)
    with pytest.raises(TypeError):
        ca.Tensor(None, ca.F32)
