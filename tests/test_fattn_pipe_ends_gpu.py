"""The pipelined tile kernel's requests behind the last key: rows of NaN bits there (a view into a longer cache), whole ranges and cut
ones, last blocks of every length, requests that start anew behind hidden keys."""
import dataclasses

import numpy as np
import pytest

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

# (head size, tile_variant, masked); 0: the planner's choice
FORMS = [(64, 0, False), (64, 0x12, False), (64, 0x11, False), (64, 0x21, False), (128, 0x11, False), (128, 0x11, True), (128, 0x21, True)]


def _behind(t, n, extra):
    """the first n rows of a tensor whose `extra` further rows are set to NaN bits"""
    buf = t.buf.copy()
    for i3 in range(t.ne[3]):
        for i2 in range(t.ne[2]):
            for i1 in range(n, n + extra):
                at = t.offset + i1 * t.nb[1] + i2 * t.nb[2] + i3 * t.nb[3]
                buf[at:at + 2 * t.ne[0]] = 0xFF
    return dataclasses.replace(t, buf=buf, ne=(t.ne[0], n, t.ne[2], t.ne[3]))


@pytest.mark.parametrize("D,variant,masked", FORMS)
@pytest.mark.parametrize("Nkv", [384, 385, 414, 449, 480, 511, 514, 705])
def test_rows_behind_the_last_key(D, variant, masked, Nkv):
    if masked and variant == 0x11 and Nkv % 2:
        Nkv += 1                                         # (odd rows are the pairs')
    Nq, extra = 90, 330
    case = make_case(seed=5000 + Nkv, D=D, Nq=Nq, Nkv=Nkv + extra, Hq=4, Hkv=2, B=2, kv_layout="thd" if Nkv % 2 else "contig")
    case["k"], case["v"] = _behind(case["k"], Nkv, extra), _behind(case["v"], Nkv, extra)
    if masked:
        j, i = np.arange(Nkv), np.arange(Nq)[:, None]
        m = np.where((j >= 300) & (j <= i * 3 + Nkv - 200), 0.0, -np.inf)
        case["mask"] = ora.from_f32(m[None, None].astype(np.float32), ora.F16)
    ref = run_oracle(case)
    for ns in (1,) if masked else (1, 2, 3):
        print("case", D, hex(variant), Nkv, ns, flush=True)
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_MMA, tile_variant=variant, n_splits=ns), ref, "%d ranges" % ns)
