"""Registers and scratch of kernels whose speed rests on them, and the wait states around inline assembly, in what the compiler
makes of the sources with the library's own flags."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from crispasr_amd import build

# 512 registers a lane and SIMD, given out in eighths: 128 leave room for four waves, 168 for three, 256 for two
F16, Q4_0, Q4_1, Q5_1, Q8_0 = 1, 2, 3, 7, 8


def _resources(source, listing):
    """{(kernel, template arguments): {"VGPRs": .., "ScratchSize": ..}} of a source's kernels; their assembly goes to `listing`"""
    res = subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-S",
                          os.path.join(build.CSRC, source), "-o", str(listing)], capture_output=True, text=True, timeout=600)
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


SOURCES = ["fattn_mma.hip", "fattn_decode.hip", "fattn_relpos.hip", "fattn_pipe.hip", "fattn_vec.hip"]


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    """(resources of all kernels, {source: its assembly's path})"""
    if not os.path.exists(build._hipcc()):
        pytest.skip("no hipcc")
    listings = {s: tmp_path_factory.mktemp("asm") / (s + ".s") for s in SOURCES}
    with ThreadPoolExecutor(len(SOURCES)) as ex:
        return {k: v for r in ex.map(_resources, SOURCES, listings.values()) for k, v in r.items()}, listings


@pytest.fixture(scope="module")
def resources(compiled):
    return compiled[0]


def _sgprs(operand):
    """the scalar registers that an operand names"""
    m = re.fullmatch(r"s(\d+)|s\[(\d+):(\d+)\]", operand)
    return set() if not m else {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def early_loads(lines):
    """memory instructions that read a scalar register fewer than five wait states after a vector instruction wrote it"""
    found, writes, clock = [], {}, 0
    for line in lines:
        line = line.split(";")[0].strip()
        if not line or line[0] in ".#" or line.endswith(":"):
            continue
        op, *rest = line.split(None, 1)
        operands = [x.split()[0] for x in rest[0].split(",") if x.strip()] if rest else []
        if op.startswith(("global_", "buffer_")):
            read = set().union(*(_sgprs(x) for x in operands))
            found += [line for r in read if clock - writes.get(r, -9) < 5]
        clock += 1 + int(operands[0], 0) if op == "s_nop" else 1
        if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")):
            writes.update({r: clock for r in _sgprs(operands[0])})
    return found


def test_early_loads_are_found():
    read = ["v_readlane_b32 s49, v255, 26", "s_mov_b32 m0, s87", "s_nop 0", "global_load_lds_dwordx4 v72, s[48:49]"]
    assert early_loads(read) == [read[3]]
    assert early_loads([read[0], "s_nop 3", read[3]]) == [read[3]]
    assert early_loads([read[0], "s_nop 4", read[3]]) == []
    assert early_loads(["v_readlane_b32 s50, v255, 26", read[3]]) == []


@pytest.mark.parametrize("source", SOURCES)
def test_no_load_reads_a_scalar_too_early(compiled, source):
    """the compiler places these wait states itself, but not between its code and inline assembly"""
    lines = open(compiled[1][source]).read().splitlines()
    assert any("global_load" in x for x in lines)
    assert early_loads(lines) == []


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


def test_short_decode_calls(resources):
    """(D, type, RAW, V8, PAD, DEEP): 64-wide f16 rows three workgroups a CU with two steps under way and four without, streamed ones four, with
    and without a mask; 128-wide f16 rows in ranges of one step a wave four"""
    forms = _forms(resources, "fattn_decode_short_kernel")
    for pad in (0, 1):
        assert forms[(64, F16, 0, 0, pad, 1)]["VGPRs"] <= 168
        assert forms[(64, F16, 0, 0, pad, 0)]["VGPRs"] <= 128
        assert forms[(128, F16, 0, 0, pad, 1)]["VGPRs"] <= 128
    masked = _forms(resources, "fattn_decode_short_masked_kernel")
    for ktype, v8 in ((Q8_0, 1), (Q4_0, 0), (Q4_1, 0), (Q5_1, 0)):
        assert forms[(64, ktype, 1, v8, 0, 0)]["VGPRs"] <= 128 and masked[(64, ktype, 1, v8, 0)]["VGPRs"] <= 128
    assert [k for f in (forms, masked) for k, r in f.items() if r["ScratchSize"]] == []


def test_short_vector_calls(resources):
    """four workgroups a CU"""
    forms = _forms(resources, "fattn_vec_short_kernel")
    assert {k[1] for k in forms} == {4, 8, 16, 32}
    assert [k for k, r in forms.items() if r["VGPRs"] > 128 or r["ScratchSize"]] == []


def test_pipelined_kernel(resources):
    """two waves a SIMD, three where a wave has one block of queries of a 64-wide head: nothing in scratch, whose waits would take the requests
    on their way in with them"""
    forms = _forms(resources, "fattn_pipe_kernel")
    assert {(k[0], k[1]) for k in forms} == {(64, 1), (64, 2), (128, 1)}
    assert [k for k, r in forms.items() if r["ScratchSize"] or r["VGPRs"] > (168 if k[:2] == (64, 1) else 256)] == []


def test_relpos_scratch(resources):
    """none, also in the forms that fill the register file"""
    forms = _forms(resources, "fattn_relpos_kernel")
    assert {k[0] for k in forms} == {64, 128}
    assert [k for k, r in forms.items() if r["ScratchSize"]] == []
