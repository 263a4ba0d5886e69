"""Unmasked F32 calls that the vector kernel takes before the tile kernel, planned without a GPU: one that needed no scratch as the tile kernel's
may overlap others on it, and has to need none as the vector kernel's."""
import ctypes
import random

import pytest

from crispasr_amd import ggml
from test_decode_ranges import _tensor


def _plan(kernel, D, H, nq, nkv):
    p = ggml._params(0.1, 0.0, 0.0, 0, kernel, 0, None)
    q, k = _tensor(ggml.F32, (D, nq, H, 1)), _tensor(ggml.F32, (D, nkv, H, 1))
    info = ggml.CPlanInfo()
    assert ggml.lib().mi355x_fattn_plan_details(ctypes.byref(q), ctypes.byref(k), ctypes.byref(k), None, ctypes.byref(p), ctypes.byref(info)) == ggml.OK
    return info


@pytest.mark.parametrize("seed", range(4))
def test_calls_without_scratch_stay_without(seed):
    r = random.Random(seed)
    moved = 0
    for _ in range(300):
        call = (r.choice([64, 128]), r.choice([1, 4, 6, 8, 12, 20]), r.choice([16, 17, 24, 31, 48]), int(2 ** r.uniform(4.2, 11)))
        auto, tile = _plan(ggml.KERNEL_AUTO, *call), _plan(ggml.KERNEL_MMA, *call)
        if tile.workspace == 0:
            assert auto.workspace == 0 and auto.n_splits == 1, call
            moved += auto.kernel == ggml.KERNEL_VEC
    assert moved > 50
