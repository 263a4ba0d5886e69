"""Counts of key ranges round which the merge inside the kernel changes its form: 4, 8 and 16 ranges are read at once, (max, sum)
pairs two to a request, and a wave merges up to four rows."""
import pytest
import torch

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_oracle, upload

pytestmark = pytest.mark.gpu

CASES = {
    # 128-wide heads, two rows a wave; the last row's last pair ends the library's scratch block
    "decode_d128": dict(seed=910, D=128, Nq=1, Nkv=2100, Hq=12, Hkv=4, ktype=ora.Q8_0),
    # 64-wide, four rows a wave that lie Hq rows apart, two chunks of 16 rows and a ragged end
    "decode_d64": dict(seed=911, D=64, Nq=19, Nkv=2100, Hq=3, Hkv=3, B=2, mask="causal"),
    # rows of 9 lanes
    "vector_d36": dict(seed=912, D=36, Nq=2, Nkv=1300, Hq=3, Hkv=3, ktype=ora.F32),
}


@pytest.mark.parametrize("ranges", [2, 4, 5, 8, 9, 16, 17, 24, 25, 33])
@pytest.mark.parametrize("name", sorted(CASES))
def test_ranges_are_merged(name, ranges):
    case = make_case(**CASES[name])
    q, k, v = upload(case["q"]), upload(case["k"]), upload(case["v"])
    m = upload(case["mask"]) if case["mask"] is not None else None
    kw = dict(kernel=ggml.KERNEL_DECODE_MMA if name.startswith("decode") else ggml.KERNEL_VEC, n_splits=ranges)
    info = ggml.flash_attn_plan_details(q, k, v, m, case["scale"], **kw)
    assert info["merge_in_kernel"] == 1
    got = [ggml.flash_attn_ext(q, k, v, m, case["scale"], **kw).numpy_f32() for _ in range(3)]      # (the counters are used again)
    assert_parity(got[0], run_oracle(case), "%s in %d ranges" % (name, ranges))
    ws = torch.empty(max(info["workspace"], 16), dtype=torch.uint8, device="cuda")
    launch = ggml.flash_attn_ext(q, k, v, m, case["scale"], workspace=ws, **kw).numpy_f32()
    for x in got:
        assert (x == launch).all()
