"""Decode calls over sequences of different lengths with more workgroups than CUs: the sequences behind the first round go by length.  Every
sequence is attended to once, whatever the mask says of its length."""
import numpy as np
import pytest

import oracle as ora
from cases import make_case
from crispasr_amd import ggml
from gpu_util import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


# a second round that is whole, in part, of one sequence; a third; first rounds of one sequence and of 64; 128 sequences and one more
@pytest.mark.parametrize("B,Hkv,gqa,D,type_,Nkv,Nq", [
    (64, 8, 1, 64, "F16", 512, 1), (33, 8, 2, 64, "F16", 519, 1), (50, 8, 1, 128, "Q8_0", 513, 2), (70, 8, 1, 64, "F16", 512, 1),
    (128, 4, 1, 64, "F16", 530, 1), (65, 4, 1, 128, "Q8_0", 512, 3), (128, 8, 1, 64, "F16", 512, 1), (129, 2, 1, 64, "F16", 512, 1),
    (20, 20, 1, 64, "F16", 600, 1), (3, 200, 1, 64, "F16", 515, 1), (2, 256, 1, 64, "F16", 512, 1), (64, 8, 1, 128, "Q4_0", 1900, 1)])
def test_every_sequence_once(B, Hkv, gqa, D, type_, Nkv, Nq):
    rng = np.random.default_rng(B * 1000 + Nkv)
    j = np.arange(Nkv)
    for what in ("lengths", "one length", "holes"):
        n = rng.integers(1, Nkv + 1, size=B) if what == "lengths" else np.full(B, Nkv - 3)
        seen = np.broadcast_to(j < n[:, None, None], (B, Nq, Nkv)).copy()
        if what == "holes":
            seen &= rng.random((B, Nq, Nkv)) < 0.3
            seen[B // 2] = False
        case = make_case(seed=4000 + B, D=D, Nq=Nq, Nkv=Nkv, Hq=Hkv * gqa, Hkv=Hkv, B=B, ktype=getattr(ora, type_))
        case["mask"] = ora.from_f32(np.where(seen, 0.0, -np.inf).astype(np.float32)[:, None], ora.F16)
        print("case", B, Hkv, D, type_, Nkv, what, flush=True)
        assert_parity(run_gpu(case, kernel=ggml.KERNEL_DECODE_MMA, n_splits=1), run_oracle(case), what)
