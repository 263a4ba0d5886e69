"""The pipelined tile kernel under masks (128-wide heads, 384 keys of a range and more): last blocks of every length, rows on and between
dwords, rows that see nothing at first or at all, bias values, ranges, references that climb, hidden rows of NaN bits."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle, upload

pytestmark = pytest.mark.gpu

FORMS = [0x11, 0x21]


def _masked(values, seed, **kw):
    """values: float32 [Bm, Hm, Nq, Nkv]"""
    case = make_case(seed=seed, D=128, Nq=values.shape[2], Nkv=values.shape[3], **kw)
    case["mask"] = ora.from_f32(values.astype(np.float32), ora.F16)
    return case


def _is_pipelined(case, variant, ns=1):
    """rows between dwords and odd key counts: the pairs' form alone"""
    t = [upload(case[n]) for n in ("q", "k", "v", "mask")]
    form = ggml.flash_attn_plan_form(*t, case["scale"], kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=ns)
    assert form == {"pipelined": int(variant == 0x21 or t[1].ne[1] % 2 == 0), "waves": 4}, form


def _run(case, variant, what, ranges=(1,)):
    print("case", hex(variant), what, flush=True)
    ref = run_oracle(case)
    for ns in ranges:
        _is_pipelined(case, variant, ns)
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=ns), ref, "%s, %d ranges" % (what, ns))


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nq,Nkv", [(1, 384), (33, 385), (64, 386), (65, 399), (129, 400), (70, 415), (128, 416), (40, 417), (66, 431), (31, 447),
                                    (97, 448), (130, 449), (200, 479), (63, 480), (34, 511), (35, 514)])
def test_last_blocks(variant, Nq, Nkv):
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    causal = np.where(j <= i + Nkv - Nq, 0.0, -np.inf)
    bias = np.random.default_rng(Nkv).normal(size=(2, 4, Nq, Nkv)) * 2.0
    bias[1, :, :, Nkv - 37:] = -np.inf
    _run(_masked(causal[None, None], 3300 + Nkv, Hq=4, Hkv=2, B=2, kv_layout="thd" if Nkv % 3 else "gap"), variant, "causal %d x %d" % (Nq, Nkv))
    _run(_masked(bias, 3400 + Nkv, Hq=4, Hkv=4, B=2), variant, "bias %d x %d" % (Nq, Nkv))


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [400, 451])
def test_rows_that_start_late(variant, Nkv):
    """first visible keys in every block, by row; rows without any; a far larger score at the end of what a row sees"""
    Nq = 150
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    late = (j >= (i * 37) % Nkv) & (i % 11 != 5)
    case = _masked(np.where(late, 0.0, -np.inf)[None, None], 3500 + Nkv, Hq=2, B=2)
    q, k = to_f32(case["q"]), to_f32(case["k"])
    k[..., 0] = np.sqrt(np.linspace(0.0, 1.0, Nkv, dtype=np.float32)) * 4.0
    q[..., 0] = 60.0 / 4.0 / case["scale"]
    q[:, :, ::3, 0] *= -1.0
    case["q"], case["k"] = ora.from_f32(q, ora.F32), ora.from_f32(k, ora.F16)
    _run(case, variant, "late rows %d" % Nkv)


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [900, 1013])
def test_ranges(variant, Nkv):
    """two ranges, the second shorter than the first: causal rows that end in either, and one length"""
    Nq = 140
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    for name, seen in (("causal", j <= i * 7), ("one length", (j < 130) & (i >= 0)), ("second range alone", j >= 600)):
        _run(_masked(np.where(seen & (i >= 0), 0.0, -np.inf)[None, None], 3600 + Nkv, Hq=4, Hkv=2), variant, "%s %d" % (name, Nkv), (1, 2))


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [500, 777])
def test_hidden_nan_rows(variant, Nkv):
    """excluded keys that hold NaN bits, scattered and at the end, by row: such rows are computed again, the others are not touched"""
    Nq = 100
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    holes = (j % 97 == 13) | (j > Nkv - 30)
    seen = ~holes & (i >= 0)
    case = _masked(np.where(seen, 0.0, -np.inf)[None, None], 3700 + Nkv, Hq=4, Hkv=2)
    ref = run_oracle(case)
    for t in (case["k"], case["v"]):
        t.buf[t.offset:].reshape(2, Nkv, -1)[:, holes] = 0xFF
    print("case", hex(variant), "hidden NaN rows", Nkv, flush=True)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1), ref)


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [384, 511, 640])
def test_extreme_mask_values(variant, Nkv):
    """the type's lowest and largest finite value in place of -inf and 0: rows of nothing else, at the start, at the end, scattered, among
    excluded keys.  V climbs from 0 to 4 with the key, so a row's result tells which keys it took.  A sum of a score and +-65504 is rounded to
    2^-8 (natural) in the oracle and to 2^-7 (log2) here, twice: no probability is off by more than 2^-6 of itself, no mean by 4 * 2^-6."""
    Nq = 70
    j, i = np.arange(Nkv), np.arange(Nq)[:, None] % 7
    low, high = -65504.0, 65504.0
    seen = j * (i + 1) % 5 < 3
    for name, m in (("lowest", np.where(i == 0, low, np.where(i == 1, np.where(j < 200, low, 0.0), np.where(i == 2, np.where(j < 200, 0.0, low),
                                np.where(i == 3, np.where(seen, low, -np.inf), np.where(i == 4, np.where(j > 300, low, -np.inf), np.where(seen, 0.0, low))))))),
                    ("largest", np.where(i < 3, np.where(j > 100 * i, high, 0.0), np.where(i < 5, np.where(seen, high, low), np.where(seen, high, -np.inf))))):
        case = _masked(np.broadcast_to(m, (1, 1, Nq, Nkv)), 3800 + Nkv, Hq=4, Hkv=2)
        case["q"] = ora.from_f32(np.clip(to_f32(case["q"]), -3, 3) * 0.05, ora.F32)
        case["v"] = ora.from_f32(np.broadcast_to((4.0 * j / Nkv)[:, None], to_f32(case["v"]).shape), ora.F16)
        ref = run_oracle(case)
        print("case", hex(variant), name, Nkv, flush=True)
        out = run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=1)
        assert np.isfinite(out).all() and np.abs(out - ref).max() <= 4 * 2.0 ** -6, (name, np.abs(out - ref).max())


@pytest.mark.parametrize("variant", FORMS)
@pytest.mark.parametrize("Nkv", [1921, 1922, 1925, 1951, 1952])
def test_a_last_range_of_fewer_keys_than_a_block(variant, Nkv):
    """six ranges of 384 keys, the sixth of 1, 2, 5, 31 and 32: its block begins in the range before, where the keys hold NaN bits and are excluded"""
    Nq = 70
    j, i = np.arange(Nkv), np.arange(Nq)[:, None]
    hidden = (j >= 1880) & (j < 1920)
    case = _masked(np.where(~hidden & (j >= i * 25) & ((j < 1920) | (i % 3 != 1)), 0.0, -np.inf)[None, None], 3900 + Nkv, Hq=4, Hkv=2)
    ref = run_oracle(case)
    for t in (case["k"], case["v"]):
        t.buf[t.offset:].reshape(2, Nkv, -1)[:, hidden] = 0xFF
    print("case", hex(variant), Nkv, "in six ranges", flush=True)
    _is_pipelined(case, variant, 6)
    assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=6), ref)
