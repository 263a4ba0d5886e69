"""Into how many key ranges the decode kernel's calls are cut, planned without a GPU: a call that was uncut uses no scratch, so it
may be captured first and overlap others, and has to stay uncut; a cut one may not outgrow the smallest scratch block."""
import ctypes
import random

import pytest

from crispasr_amd import ggml

TYPES = {"f16": (ggml.F16, 2), "q8_0": (ggml.Q8_0, 34 / 32), "q4_0": (ggml.Q4_0, 18 / 32), "q5_1": (ggml.Q5_1, 24 / 32)}


def _tensor(type_, ne, data=4096):
    t = ggml.CTensor()
    t.data, t.type = data, type_
    nb = [ggml.TYPE_SIZE[type_], ggml.row_size(type_, ne[0])]
    for n in ne[1:3]:
        nb.append(nb[-1] * n)
    t.ne, t.nb = (ctypes.c_int64 * 4)(*ne), (ctypes.c_size_t * 4)(*nb)
    return t


def _plan(ktype, hd, hq, hkv, B, nq, nkv, masked):
    p = ggml._params(0.1, 0.0, 0.0, 0, ggml.KERNEL_DECODE_MMA, 0, None)
    q, k = _tensor(ggml.F32, (hd, nq, hq, B)), _tensor(TYPES[ktype][0], (hd, nkv, hkv, B))
    m = _tensor(ggml.F16, (nkv, nq, 1, 1)) if masked else None
    info = ggml.CPlanInfo()
    rc = ggml.lib().mi355x_fattn_plan_details(*(ctypes.byref(x) if x is not None else None for x in (q, k, k, m)), ctypes.byref(p), ctypes.byref(info))
    assert rc == ggml.OK
    return info.n_splits, info.workspace


def _was_cut(ktype, hd, hq, hkv, B, nq, nkv, cus=256):
    """the count that was chosen before the pricing by steps, ports and batches"""
    gqa = hq // hkv
    groups, min_keys = hkv * B * ((nq * gqa + 15) // 16), 128 if hd <= 64 else 64
    ns = min(2 * cus // groups, (nkv + min_keys // 2) // min_keys)
    if ns < 2:
        return 1
    hbm = max(0.0, (hkv * B * nkv * 2 * hd * TYPES[ktype][1] - 8e6) / 5e6)
    price = {}
    for n in range(1, ns + 1):
        keys = ((nkv + n - 1) // n + 31) // 32 * 32
        if (nkv + keys - 1) // keys == n:
            chain = max(1.0, keys / 128) * (0.7 if hd <= 64 else 1.3) * max(1.0, groups * n / cus)
            price[n] = max(chain, hbm) + (1 + n * (0.25 + 0.017 * min(16, nq * gqa)) if n > 1 else 0)
    return max(n for n in price if price[n] <= min(price.values()) * 1.10)


@pytest.mark.parametrize("seed", range(8))
def test_uncut_calls_stay_uncut(seed):
    r = random.Random(seed)
    uncut = 0
    for _ in range(300):
        hd, hq, hkv = r.choice([(128, 32, 8), (128, 16, 8), (128, 8, 8), (64, 16, 16), (64, 32, 8), (64, 20, 20), (64, 6, 6)])
        call = (r.choice(sorted(TYPES)), hd, hq, hkv, r.choice([1, 1, 2, 3, 8, 17, 40, 64]), r.choice([1, 1, 2, 5, 16, 40]), int(2 ** r.uniform(4, 14)))
        ns, need = _plan(*call, masked=r.random() < 0.5)
        before, part = _was_cut(*call), call[2] * call[4] * call[5] * (hd + 2) * 4
        assert (ns > 1) <= (before > 1), (call, ns, before)
        assert need <= max(4 << 20, 2 * part + 512), (call, ns, need)
        assert ns == 1 or need >= ns * part
        uncut += before == 1
    assert 50 < uncut < 250


def _plan_in(room, ktype, hd, hq, hkv, B, nq, nkv):
    """the ranges of the call on a caller's workspace of `room` bytes"""
    p = ggml._params(0.1, 0.0, 0.0, 0, ggml.KERNEL_DECODE_MMA, 0, None)
    p.workspace, p.workspace_size = 4096, room
    q, k = _tensor(ggml.F32, (hd, nq, hq, B)), _tensor(TYPES[ktype][0], (hd, nkv, hkv, B))
    info = ggml.CPlanInfo()
    assert ggml.lib().mi355x_fattn_plan_details(ctypes.byref(q), ctypes.byref(k), ctypes.byref(k), None, ctypes.byref(p), ctypes.byref(info)) == ggml.OK
    return info


@pytest.mark.parametrize("seed", range(4))
def test_workspaces_of_the_former_sizes_still_do(seed):
    """a caller's workspace that holds the ranges a call was once cut into, and fewer than it is cut into now, takes as many as fit"""
    r = random.Random(100 + seed)
    held = 0
    for _ in range(300):
        hd, hq, hkv = r.choice([(128, 32, 8), (128, 16, 8), (64, 16, 16), (64, 32, 8), (64, 20, 20), (64, 6, 6)])
        call = (r.choice(sorted(TYPES)), hd, hq, hkv, r.choice([1, 2, 8, 17, 40]), r.choice([1, 1, 5, 16]), int(2 ** r.uniform(8, 14)))
        ns, need = _plan(*call, masked=False)
        before, part = _was_cut(*call), call[2] * call[4] * call[5] * (hd + 2) * 4
        for room in (before * part, before * part + part // 2, need - 1, need):
            info = _plan_in(room, *call)
            assert info.workspace == need
            if ns == 1 or room >= need:
                assert info.n_splits == ns, (call, room, info.n_splits, ns)
            elif room >= before * part:
                assert 2 <= info.n_splits < ns and info.n_splits * part <= room, (call, room, info.n_splits, ns)
                assert info.n_splits * info.keys_per_split >= call[6] > (info.n_splits - 1) * info.keys_per_split and info.keys_per_split % 32 == 0
                held += 1
    assert held > 50
