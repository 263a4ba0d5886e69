"""The pipelined tile kernel under masks that hide keys ahead of the first visible one (windows, padding on the left, several sequences
in a row): where the walk starts, rows that see their first key late, and what such a call takes."""
import numpy as np
import pytest
import torch

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle, upload

pytestmark = pytest.mark.gpu

FORMS = [0x11, 0x21]


def _run(seen, seed, variant, what, ranges=(1,), nan=False, **kw):
    """seen: bool [Nq, Nkv] or [B, 1, Nq, Nkv]"""
    seen = seen if seen.ndim == 4 else seen[None, None]
    case = make_case(seed=seed, D=128, Nq=seen.shape[2], Nkv=seen.shape[3], Hq=4, Hkv=2, B=seen.shape[0], **kw)
    case["mask"] = ora.from_f32(np.where(seen, 0.0, -np.inf).astype(np.float32), ora.F16)
    ref = run_oracle(case)
    if nan:                                            # keys that nobody sees hold NaN bits
        unseen = ~seen.any(axis=(0, 1, 2))
        for t in (case["k"], case["v"]):
            t.buf[t.offset:].reshape(2 * seen.shape[0], seen.shape[3], -1)[:, unseen] = 0xFF
    print("case", hex(variant), what, flush=True)
    for ns in ranges:
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=ns), ref, "%s, %d ranges" % (what, ns))


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [450, 777, 1030])
def test_first_visible_key(variant, Nkv):
    """one first key for all queries, round the first tiles that are left out (four of 64 keys) and the last keys of the row"""
    Nq = 70
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    for first in (0, 63, 64, 255, 256, 257, 300, 319, 320, 352, 384, Nkv - 65, Nkv - 33, Nkv - 32, Nkv - 31, Nkv - 1):
        _run((j >= first) & (i >= 0), 3900 + first, variant, "first key %d of %d" % (first, Nkv), nan=first % 2 == 1)


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nq,Nkv", [(200, 600), (333, 1021), (130, 1200)])
def test_windows_and_sequences(variant, Nq, Nkv):
    j, i = np.arange(Nkv), np.arange(Nq)[:, None] + Nkv - Nq
    for what, seen in (("window", (j <= i) & (j > i - 100)),
                       ("sequences in a row", (j <= i) & (j * 5 // Nkv == i * 5 // Nkv)),
                       ("a prefix and a window", (j <= i) & ((j > i - 70) | (j < 30))),
                       ("windows that move left", (j >= Nkv - 40 - i) & (j < Nkv + 60 - i)),
                       ("rows without a key", (j <= i) & (j > i - 100) & (i % 3 != 1)),
                       ("a hole", (j < 100) | (j > 450 + i % 50))):
        _run(seen, 4000 + Nkv, variant, "%s, %d x %d" % (what, Nq, Nkv), ranges=(1, 2) if Nkv >= 900 else (1,), nan=what == "window")
    n = np.array([0, Nkv // 3, Nkv - 5])[:, None, None, None]
    _run((j >= n) & (i >= 0), 4100 + Nkv, variant, "sequences padded on the left, %d x %d" % (Nq, Nkv))


@pytest.mark.parametrize("variant", FORMS)
def test_late_rows_with_large_scores(variant):
    """rows whose first keys come in every block, with references far below and above zero and scores that climb past f16's range"""
    Nq, Nkv = 140, 900
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    seen = j >= 300 + (i * 37) % 580
    case = make_case(seed=4200, D=128, Nq=Nq, Nkv=Nkv, Hq=2, Hkv=2)
    case["mask"] = ora.from_f32(np.where(seen, 0.0, -np.inf).astype(np.float32)[None, None], ora.F16)
    q, k = to_f32(case["q"]), to_f32(case["k"])
    k[..., 0] = np.sqrt(np.linspace(0.2, 1.0, Nkv, dtype=np.float32)) * 4.0
    q[..., 0] = 60.0 / 4.0 / case["scale"]
    q[:, :, ::3, 0] *= -1.0
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, ora.F16)
    print("case", hex(variant), "late rows", flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), run_oracle(case))


def _us(q, k, v, m, out, scale):
    best = 1e30
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            ggml.flash_attn_ext(q, k, v, m, scale, out=out)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 100.0)
    return best


def test_hidden_keys_cost_less_than_visible_ones():
    """2048 queries x 8 heads (two waves a query block) and 32 heads (one), against the same call with every key visible.  A window of 256 and a
    hidden first half leave at most an eighth and a half of the keys to walk: 0.45 to 0.8 of the time.  Walked from the first key on they take
    1.04 to 1.1 times it with 8 heads."""
    N = 2048
    j, i = np.arange(N), np.arange(N)[:, None]
    for Hq, Hkv in ((8, 8), (32, 8)):
        case = make_case(seed=4300, D=128, Nq=N, Nkv=N, Hq=Hq, Hkv=Hkv)
        q, k, v = upload(case["q"]), upload(case["k"]), upload(case["v"])
        out = ggml.Tensor.empty(ggml.F32, (128, Hq, N, 1))
        us = {}
        for what, seen in (("all", (j >= 0) & (i >= 0)), ("window", (j <= i) & (j > i - 256)), ("second half", (j >= N // 2) & (i >= 0)),
                           ("four sequences", (j <= i) & (j * 4 // N == i * 4 // N))):
            m = upload(ora.from_f32(np.where(seen, 0.0, -np.inf).astype(np.float32)[None, None], ora.F16))
            us[what] = _us(q, k, v, m, out, case["scale"])
        print("%d heads" % Hq, {w: round(t, 1) for w, t in us.items()}, flush=True)
        assert max(us["window"], us["four sequences"], us["second half"]) < 0.92 * us["all"], us
