"""The pipelined tile kernel's forms of 128-wide heads as calls that leave the kernel's form to the library reach them: masked ranges from 64 keys
(pairs of waves) and from 128 (waves of their own), unmasked pairs, heads padded to 128: block and step counts of every remainder, rows of masks
between dwords, hidden rows, keys that rows see late, ranges, NaN bits behind the last key."""
import numpy as np
import pytest

from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle, upload
from test_fattn_pipe_ends_gpu import _behind
from test_fattn_pipe_mask_gpu import _masked

pytestmark = pytest.mark.gpu


def _run(case, what, piped=1, ns=1):
    print("case", what, flush=True)
    t = [upload(case[n]) for n in ("q", "k", "v")] + [upload(case["mask"]) if case["mask"] is not None else None]
    form = ggml.flash_attn_plan_form(*t, case["scale"], kernel=ggml.KERNEL_MMA, n_splits=ns)
    assert form["pipelined"] == piped, form
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, n_splits=ns), run_oracle(case), what)


def _masks(Nq, Nkv, heads, batch):
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    causal = np.where((j <= i + Nkv - Nq) & (i % 13 != 7), 0.0, -np.inf)[None, None]
    late = np.where((j >= (i * 37) % Nkv) & (i % 11 != 5), 0.0, -np.inf)[None, None]
    bias = np.random.default_rng(Nkv).normal(size=(batch, heads, Nq, Nkv)) * 2.0
    bias[0, :, :, Nkv - 21:] = -np.inf
    return (("causal", causal), ("late", late), ("bias", bias))


@pytest.mark.parametrize("Nq,Nkv,piped", [(5, 63, 0), (64, 64, 1), (33, 65, 1), (100, 95, 1), (65, 96, 1), (31, 97, 1), (128, 127, 1), (129, 128, 1), (70, 130, 1),
                                          (200, 159, 1), (63, 192, 1), (66, 193, 1), (130, 255, 1), (34, 322, 1), (257, 383, 1)])
def test_masked_pairs(Nq, Nkv, piped):
    for what, m in _masks(Nq, Nkv, 4, 2):
        case = _masked(m, 6100 + Nkv, Hq=4, Hkv=2, B=2, kv_layout="thd" if Nkv % 3 else "gap")
        _run(case, "%s %d x %d" % (what, Nq, Nkv), piped)


# (more workgroups of 64 queries than CUs: 300 heads)
@pytest.mark.parametrize("Nq,Nkv,piped", [(40, 127, 0), (40, 126, 0), (33, 128, 1), (40, 129, 0), (64, 130, 1), (65, 158, 1), (20, 192, 1), (130, 222, 1), (70, 382, 1)])
def test_masked_waves_of_their_own(Nq, Nkv, piped):
    for what, m in _masks(Nq, Nkv, 1, 1):
        _run(_masked(m, 6200 + Nkv, Hq=20, Hkv=10, B=15), "%s %d x %d" % (what, Nq, Nkv), piped)


@pytest.mark.parametrize("D", [128, 96, 80])
@pytest.mark.parametrize("Nq,Nkv,piped", [(1, 1, 0), (40, 31, 0), (70, 32, 0), (63, 33, 1), (64, 64, 1), (65, 95, 1), (100, 97, 1), (31, 128, 1), (130, 160, 1),
                                          (70, 191, 1), (33, 300, 1), (129, 513, 1),
                                          # half a tile of keys, and few rows of one tile or three, are the tile kernel's
                                          (48, 64, 0), (49, 64, 1), (5, 65, 1), (24, 128, 1), (24, 129, 0), (25, 129, 1), (24, 192, 0), (7, 193, 1)])
def test_plain_pairs(D, Nq, Nkv, piped):
    case = make_case(seed=6300 + Nkv, D=D, Nq=Nq, Nkv=Nkv, Hq=4, Hkv=2, B=2, q_layout="thd", kv_layout="thd" if Nkv % 2 else "gap")
    _run(case, "plain %d %d x %d" % (D, Nq, Nkv), piped)


@pytest.mark.parametrize("ns,Nkv", [(2, 200), (3, 390), (4, 420), (2, 1000)])
def test_ranges(ns, Nkv):
    _run(make_case(seed=6400 + Nkv, D=128, Nq=70, Nkv=Nkv, Hq=4, Hkv=2), "plain %d" % Nkv, ns=ns)
    for what, m in _masks(70, Nkv, 4, 1):
        _run(_masked(m, 6400 + Nkv, Hq=4, Hkv=2), "%s %d in %d" % (what, Nkv, ns), ns=ns)


@pytest.mark.parametrize("Nkv", [64, 90, 129, 250])
def test_nan_bits_behind_the_last_key(Nkv):
    for D in (128, 80):
        case = make_case(seed=6500 + Nkv, D=D, Nq=90, Nkv=Nkv + 600, Hq=4, Hkv=2, kv_layout="thd" if Nkv % 4 else "contig")
        case["k"], case["v"] = _behind(case["k"], Nkv, 600), _behind(case["v"], Nkv, 600)
        _run(case, "plain %d %d" % (D, Nkv))
