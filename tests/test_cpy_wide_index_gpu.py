"""Launches of 2^31 lanes and more, where the copy kernels index with 64 bits: one such call equals, byte for byte, the same
rows in four calls that are below the line (and whose kernels the other tests hold to the oracle).  The sources are windows
of a small buffer that overlap, no two alike, so that only the destinations take memory (up to 69 GB)."""
import pytest
import torch

import crispasr_amd as ca
import oracle as ora

pytestmark = pytest.mark.gpu

BLOCKS = [ora.Q8_0, ora.Q4_0, ora.Q4_1, ora.Q5_0, ora.Q5_1]
LINE = 1 << 31
U0, N1, N2 = 1031, 7, 64                           # units along dimension 0 (a prime), rows, heads


def room(nbytes):
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < nbytes + (4 << 30):
        pytest.skip("needs %d GB of device memory" % (nbytes >> 30))


def noise(type_, nbytes, seed):
    """finite values of a type: normal F32, or bytes whose halves have exponents below f16's upper half"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if type_ == ora.F32:
        return torch.randn((nbytes + 3) // 4, generator=g, device="cuda").view(torch.uint8)
    return torch.randint(0, 256, (nbytes,), generator=g, device="cuda", dtype=torch.uint8) & 0xBF


def windows(type_, ne, step, lead, seed):
    """a tensor whose sequences (dimension 3) start `step` bytes apart in one buffer"""
    rs = ora.row_size(type_, ne[0])
    slab = rs * ne[1] * ne[2]
    return ca.Tensor(noise(type_, lead + slab + step * ne[3], seed), type_, ne, (ora.TYPE_SIZE[type_], rs, rs * ne[1], step), lead)


def sequences(t, first, n):
    return ca.Tensor(t.buf, t.type, t.ne[:3] + (n,), t.nb, t.offset + first * t.nb[3])


def compare(n3, slab, lead, big, fill):
    """big: bytes of the one call, behind `lead`; fill(first, n, buffer) makes sequences first .. first + n - 1"""
    quarter = (n3 + 3) // 4
    piece = torch.empty(lead + slab * quarter, dtype=torch.uint8, device="cuda")
    for first in range(0, n3, quarter):
        n = min(quarter, n3 - first)
        fill(first, n, piece)
        want, got = piece[lead:lead + slab * n], big[lead + slab * first:lead + slab * (first + n)]
        for at in range(0, slab * n, 1 << 30):                     # (a comparison makes a byte for every one)
            assert torch.equal(got[at:at + (1 << 30)], want[at:at + (1 << 30)]), (first, at)


# (source, destination, elements a unit, lanes a unit, bytes the rows lie off 16)
PLAIN = [(s, d, 8 if not off else 1, 1, off) for s in (ora.F32, ora.F16) for d in (ora.F32, ora.F16) for off in (0, 4)]
TO_BLOCKS = [(ora.F32, t, 32, 4, off) for t in BLOCKS for off in (0, 4)]
FROM_BLOCKS = [(t, ora.F32, 32, 4, off) for t in BLOCKS for off in (0, 4)]
MOVED = [(t, t, 32, ora.TYPE_SIZE[t] // 2, 0) for t in BLOCKS]


@pytest.mark.parametrize("stype,dtype,unit,lanes,off", PLAIN + TO_BLOCKS + FROM_BLOCKS + MOVED)
def test_copies(stype, dtype, unit, lanes, off):
    n3 = LINE // (U0 * N1 * N2 * lanes) + 1
    ne = (U0 * unit, N1, N2, n3)
    slab = ora.row_size(dtype, ne[0]) * N1 * N2
    room(slab * (n3 + n3 // 4 + 1))
    src = windows(stype, ne, 32 * 37 if stype not in BLOCKS else 37 * ora.TYPE_SIZE[stype], off, 7100 + stype + 16 * dtype)
    print("copy", stype, dtype, ne, off, flush=True)

    def into(buf, part, flat=False):
        shape = part.ne if not flat else (part.ne[0] * N1, N2, part.ne[3], 1)
        return ca.cpy(part, ca.Tensor(buf, dtype, shape, None, off))

    big = torch.empty(off + slab * n3, dtype=torch.uint8, device="cuda")
    for flat in (False, True):                                     # a destination of the same shape, and of another
        big.fill_(0xA5)
        into(big, src, flat)
        compare(n3, slab, off, big, lambda first, n, buf: into(buf, sequences(src, first, n)))


@pytest.mark.parametrize("dtype,unit,lanes,off", [(t, 32, 4, off) for t in BLOCKS for off in (0, 4)] +
                         [(t, 8 if not off else 1, 1, off) for t in (ora.F32, ora.F16) for off in (0, 4)])
def test_set_rows(dtype, unit, lanes, off):
    n3 = LINE // (U0 * N1 * N2 * lanes) + 1
    ne = (U0 * unit, N1, N2, n3)
    slab = ora.row_size(dtype, ne[0]) * N1 * N2
    room(slab * (n3 + n3 // 4 + 1))
    src = windows(ora.F32, ne, 32 * 37, off, 7300 + dtype)
    g = torch.Generator().manual_seed(7300)
    idx = torch.stack([torch.randperm(N1, generator=g) for _ in range(N2)]).view(1, N2, N1).to("cuda")
    print("set_rows", dtype, ne, off, flush=True)
    big = torch.full((off + slab * n3,), 0xA5, dtype=torch.uint8, device="cuda")
    ca.set_rows(ca.Tensor(big, dtype, ne, None, off), src, idx)

    def fill(first, n, buf):
        part = sequences(src, first, n)
        ca.set_rows(ca.Tensor(buf, dtype, part.ne, None, off), part, idx)

    compare(n3, slab, off, big, fill)


# F16 copies of K and V ahead of the tile kernel: 8 elements a lane, both tensors in one launch
@pytest.mark.parametrize("D,ktype,vtype", [(64, ora.F32, ora.F32)] + [(64, t, t) for t in BLOCKS] +
                         [(64, ora.Q8_0, ora.F16), (48, ora.F16, ora.F16)])
def test_attention_over_converted_caches(D, ktype, vtype):
    H, Nq, Nkv = 64, 128, 1024
    B = LINE // (2 * 8 * Nkv * H) + 1                              # (heads of 48 are copied into rows of 64)
    room((2 * 64 * Nkv * H * B * 2) * 5 // 4 + 4 * D * H * Nq * B * 3 // 2)
    q = windows(ora.F32, (D, Nq, H, B), 5 * 4 * D, 0, 7501)
    k = windows(ktype, (D, Nkv, H, B), 5 * ora.row_size(ktype, D), 0, 7502)
    v = windows(vtype, (D, Nkv, H, B), 5 * ora.row_size(vtype, D), 0, 7503)
    scale = 1.0 / D ** 0.5
    plans = []

    def attend(first, n, buf):
        qs, ks, vs = (sequences(t, first, n) for t in (q, k, v))
        plan = ca.ggml.flash_attn_plan_details(qs, ks, vs, None, scale)
        assert plan["kv_to_f16"]
        plans.append(tuple(v for f, v in plan.items() if f != "workspace"))
        ws = torch.empty(ca.ggml.flash_attn_workspace_size(qs, ks, vs, None, scale), dtype=torch.uint8, device="cuda")
        ca.flash_attn_ext(qs, ks, vs, None, scale, out=ca.Tensor(buf, ora.F32, (D, H, Nq, n)), workspace=ws)

    print("attention", D, ktype, vtype, B, flush=True)
    slab = 4 * D * H * Nq
    big = torch.full((slab * B,), 0xFF, dtype=torch.uint8, device="cuda")
    attend(0, B, big)
    compare(B, slab, 0, big, attend)
    assert len(set(plans)) == 1, plans
