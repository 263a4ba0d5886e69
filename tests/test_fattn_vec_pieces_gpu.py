"""The vector kernel's short form (no mask, F32 rows or f16 rows that the decode kernel does not take, one row a (head, sequence) or one
sequence): rows that end inside a lane's eight elements, every number of lanes a row, whole and 8-byte rows, one range and several, ends of
steps, broadcast sequences, infinities in the last key, NaN bits behind it - and calls next to its rule, which keep the general form."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case, to_f32
from crispasr_amd import ggml
from gpu_util import assert_parity, kernel_form, run_gpu, run_oracle
from test_fattn_pipe_ends_gpu import _behind

pytestmark = pytest.mark.gpu


def _run(case, ns, form=ggml.FORM_SHORT):
    assert kernel_form(case, kernel=ggml.KERNEL_VEC, n_splits=ns) == form
    return run_gpu(case, kernel=ggml.KERNEL_VEC, n_splits=ns)


@pytest.mark.parametrize("ktype", [ora.F32, ora.F16])
@pytest.mark.parametrize("D", [8, 20, 32, 36, 52, 64, 68, 72, 100, 128, 132, 256])
def test_head_sizes(D, ktype):
    for Nkv, ns in ((1, 1), (127, 1), (129, 1), (375, 3), (515, 2), (700, 0)):
        case = make_case(seed=6100 + D + Nkv, D=D, Nq=1, Nkv=Nkv, Hq=3, ktype=ktype, kv_layout="thd" if Nkv % 2 else "gap")
        print("case", D, ktype, Nkv, ns, flush=True)
        assert_parity(_run(case, ns), run_oracle(case))


@pytest.mark.parametrize("ktype,D,Nq,B,Bk,q_layout", [
    (ora.F32, 36, 5, 1, 1, "thd"), (ora.F16, 36, 24, 1, 1, "thd"), (ora.F32, 52, 1, 4, 4, "contig"), (ora.F32, 36, 1, 3, 1, "thd"),
    (ora.F16, 52, 1, 4, 1, "contig"), (ora.F32, 64, 2, 1, 1, "thd"),
    (ora.F32, 36, 2, 3, 3, "thd"), (ora.F16, 36, 2, 2, 1, "contig")])              # (several rows of several sequences: the general form)
def test_rows_and_sequences(ktype, D, Nq, B, Bk, q_layout):
    for ns in (1, 4):
        case = make_case(seed=6200 + D + Nq + B, D=D, Nq=Nq, Nkv=333, Hq=6, B=B, Bk=Bk, ktype=ktype, q_layout=q_layout, kv_layout="thd")
        print("case", ktype, D, Nq, B, Bk, ns, flush=True)
        assert_parity(_run(case, ns, ggml.FORM_GENERAL if Nq > 1 and B > 1 else ggml.FORM_SHORT), run_oracle(case))


@pytest.mark.parametrize("kw", [dict(Hkv=2), dict(mask="random_inf"), dict(softcap=20.0)])
def test_calls_next_to_the_rule(kw):
    case = make_case(seed=6300, D=36, Nq=1, Nkv=300, Hq=4, ktype=ora.F32, **kw)
    assert_parity(_run(case, 2, ggml.FORM_GENERAL), run_oracle(case))


@pytest.mark.parametrize("ktype,D,Nkv", [(ora.F32, 36, 100), (ora.F32, 64, 375), (ora.F16, 36, 130), (ora.F16, 52, 97)])
def test_nan_bits_behind_the_last_key(ktype, D, Nkv):
    case = make_case(seed=6400 + Nkv, D=D, Nq=1, Nkv=Nkv + 40, Hq=4, ktype=ktype, kv_layout="thd")
    case["k"], case["v"] = _behind(case["k"], Nkv, 40), _behind(case["v"], Nkv, 40)
    for ns in (1, 3):
        assert_parity(_run(case, ns), run_oracle(case))


@pytest.mark.parametrize("ktype", [ora.F32, ora.F16])
def test_infinite_values_of_the_last_key(ktype):
    case = make_case(seed=6500, D=36, Nq=1, Nkv=130, Hq=2, ktype=ktype)
    v = to_f32(case["v"])
    v[..., -1, 3] = np.inf
    case["v"] = ora.from_f32(v, ktype)
    got, ref = _run(case, 1), run_oracle(case)
    assert np.isposinf(ref[..., 3]).all() and np.isposinf(got[..., 3]).all()
    keep = np.arange(36) != 3
    assert_parity(got[..., keep], ref[..., keep])
