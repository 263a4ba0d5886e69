"""Registers and scratch of kernels whose speed rests on them, as the compiler reports them for the library's own flags."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from crispasr_amd import build

# 512 registers a lane and SIMD, given out in eighths: 128 leave room for four waves, 168 for three, 256 for two
F16, Q4_0, Q4_1, Q5_1, Q8_0 = 1, 2, 3, 7, 8


def _resources(source):
    """{(kernel, template arguments): {"VGPRs": .., "ScratchSize": ..}} of a source's kernels"""
    res = subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                          os.path.join(build.CSRC, source), "-o", os.devnull], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr[-2000:]
    out, name = {}, None
    for line in res.stderr.splitlines():
        m = re.search(r"remark:\s+(Function Name|VGPRs|ScratchSize)(?: \[[^\]]*\])?: (\S+)", line)
        if not m:
            continue
        if m[1] == "Function Name":
            kernel = re.match(r"_ZN12_GLOBAL__N_1\d+([a-z0-9_]+)I((?:L[ib]\d+E)+)E", m[2])
            name = (kernel[1], tuple(int(x) for x in re.findall(r"L[ib](\d+)E", kernel[2]))) if kernel else None
        elif name:
            out.setdefault(name, {})[m[1]] = int(m[2])
    return out


def test_matrix_instructions_are_the_compilers():
    """none in inline assembly, nor moves of their results: the wait states between the two are the compiler's to place"""
    for f in sorted(os.listdir(build.CSRC)):
        if f.endswith((".hip", ".h")):
            code = open(os.path.join(build.CSRC, f)).read()
            for m in re.finditer(r'\basm\b[^;]*;', re.sub(r"//.*", "", code)):
                assert not re.search(r"v_mfma|v_smfmac|v_mov_b32|v_accvgpr", m[0]), (f, m[0])


@pytest.fixture(scope="module")
def resources():
    if not os.path.exists(build._hipcc()):
        pytest.skip("no hipcc")
    sources = ["fattn_mma.hip", "fattn_decode.hip", "fattn_relpos.hip"]
    with ThreadPoolExecutor(len(sources)) as ex:
        return {k: v for r in ex.map(_resources, sources) for k, v in r.items()}


def _forms(resources, kernel):
    return {args: r for (name, args), r in resources.items() if name == kernel}


def test_decode_without_a_mask(resources):
    """64-wide f16 rows, whole heads and padded ones: four workgroups a CU"""
    forms = _forms(resources, "fattn_decode_kernel")
    for pad in (0, 1):
        assert forms[(64, F16, 0, 0, 0, pad)]["VGPRs"] <= 128
    assert all(r["ScratchSize"] == 0 for r in forms.values())


def test_decode_under_a_mask(resources):
    """64-wide streamed caches: the look at the mask takes no workgroup from a CU"""
    forms = _forms(resources, "fattn_decode_kernel")
    assert forms[(64, Q8_0, 1, 1, 1, 0)]["VGPRs"] <= 128
    for ktype in (Q4_0, Q4_1, Q5_1):
        assert forms[(64, ktype, 1, 1, 0, 0)]["VGPRs"] <= 128


def test_tile_kernel_under_a_mask(resources):
    """f16 rows moved straight to LDS: no form keeps anything in scratch"""
    forms = {k: r for k, r in _forms(resources, "fattn_mma_kernel").items() if k[6]}
    assert {(k[0], k[1]) for k in forms} == {(64, 1), (64, 2), (128, 1)}
    assert [k for k, r in forms.items() if r["ScratchSize"]] == []


def test_relpos_scratch(resources):
    """none inside the step loop; the forms that fill the register file hold up to three registers of the epilogue there"""
    forms = _forms(resources, "fattn_relpos_kernel")
    assert {k[0] for k in forms} == {64, 128}
    for args, r in forms.items():
        assert r["ScratchSize"] <= (16 if args[0] == 128 else 0), (args, r)
