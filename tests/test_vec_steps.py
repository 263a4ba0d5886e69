"""Unmasked F32 calls that the vector kernel takes before the tile kernel, planned without a GPU: one that needed no scratch as the tile kernel's
may overlap others on it, and has to need none as the vector kernel's."""
import ctypes
import random

import pytest

from crispasr_amd import ggml
from test_decode_ranges import _tensor


def _plan(kernel, D, H, nq, nkv, room=None):
    p = ggml._params(0.1, 0.0, 0.0, 0, kernel, 0, None)
    if room is not None:
        p.workspace, p.workspace_size = 4096, room
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


@pytest.mark.parametrize("D", [32, 48, 80, 96])
def test_workspaces_that_held_the_padded_copies_still_do(D):
    """one or two heads of many rows, whose partials take more than the copies: whole on a workspace of the copies' size, and refused on
    a smaller one, as the tile kernel's call was"""
    r = random.Random(D)
    held = 0
    for _ in range(3000):
        H = r.choice([1, 1, 1, 2])
        rows = r.randint(200, 1024)
        call = (D, H, rows // H, r.randint(150, 600))
        auto, tile = _plan(ggml.KERNEL_AUTO, *call), _plan(ggml.KERNEL_MMA, *call)
        if auto.kernel != ggml.KERNEL_VEC or auto.workspace <= tile.workspace or call[1] * call[2] * call[3] < 100000:
            continue
        assert tile.head_pad
        whole = _plan(ggml.KERNEL_AUTO, *call, room=tile.workspace)
        assert (whole.kernel, whole.n_splits, whole.keys_per_split, whole.workspace, whole.merge_in_kernel) == (ggml.KERNEL_VEC, 1, call[3], 0, 0), call
        assert _plan(ggml.KERNEL_AUTO, *call, room=tile.workspace - 16).workspace == auto.workspace
        held += 1
    assert held > 20
