"""Registers of the attention kernels, as the compiler reports them: a kernel that spills pays for it on every page
it walks.  No device is needed."""
import functools
import os
import re
import shutil
import subprocess
import tempfile

import pytest

from breccia_amd import build


@functools.lru_cache(maxsize=None)
def compiled(source):
    """-> what the compiler says of each kernel's resources, and its assembly"""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    with tempfile.TemporaryDirectory() as tmp:
        asm = os.path.join(tmp, "kernels.s")
        proc = subprocess.run([hipcc] + build.HIP_FLAGS + build.FILE_FLAGS.get(source, []) +
                              ["--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                               "-I", os.path.join(build.HERE, "..", "include"), "-S", os.path.join(build.CSRC, source),
                               "-o", asm], capture_output=True, text=True)
        assert proc.returncode == 0, proc.stderr[-2000:]
        with open(asm) as f:
            return proc.stderr, f.read()


def scratch_of_kernels(source):
    return dict(re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", compiled(source)[0], re.S))


def test_decode_kernels_do_not_spill():
    scratch = scratch_of_kernels("decode_attn_mfma.hip")
    # f16, q8_0 V, int8: the fused step, the step of a recorded plan, dense, a selection list; f16 again for few entries
    decode = {k: int(v) for k, v in scratch.items() if re.search(r"decode_attn_(mfma\w*|few)_kernelI", k)}
    steps = [k for k in decode if re.search(r"_kernelILb1E", k)]  # <STEP, ...>: the template's first argument
    assert len(decode) == 15 and len(steps) == 7, sorted(scratch)
    # int8 lists: 24 bytes a lane, a quad that a page fetches back once and a dword on a rare path
    int8_list = [k for k in decode if "decode_attn_mfma_i8h_kernelILb0ELb0ELb1E" in k]
    assert len(int8_list) == 1 and decode.pop(int8_list[0]) <= 24, scratch
    assert not any(decode.values()), decode


def test_chunk_kernels_do_not_spill():
    # 512 registers of a lone wave: f16 with one tile a wave and two, both quantised layouts, cut and not
    scratch = scratch_of_kernels("prefill_attn.hip")
    chunk = {k: int(v) for k, v in scratch.items() if "prefill_attn_kernel" in k}
    assert len(chunk) == 7, sorted(scratch)
    assert not any(chunk.values()), chunk


def test_chunk_kernels_hold_little_beside_q_in_the_upper_registers():
    # Before a wave of 512 registers spills to memory it moves values through its upper half, which the VALU cannot read.
    # q of two tiles takes 128 there.  Quantised pages: what else lives there is needed once a step or less, fewer than 72
    # values; more, and codes that were just requested are among them (and waited for).
    remarks, text = compiled("prefill_attn.hip")
    upper = {k: int(v) for k, v in re.findall(r"Function Name: (\S+).*?AGPRs: (\d+)", remarks, re.S) if "prefill_attn_kernel" in k}
    assert len(upper) == 7, sorted(upper)
    for name, count in upper.items():
        layout, tiles = map(int, re.search(r"prefill_attn_kernelILi(\d)ELi(\d)", name).groups())
        body = text[text.index("\n" + name + ":"):]
        back = len(re.findall(r"^\s+v_accvgpr_read", body[:body.index(".Lfunc_end")], re.M))
        assert (count, back) == (0, 0) if tiles == 1 else (count, back) == (128, 0) if layout == 0 else count < 128 + 72, (name, count, back)


@pytest.mark.parametrize("source", ["decode_attn_mfma.hip", "prefill_attn.hip", "kv_move.hip", "select.hip"])
def test_kernels_know_which_memory_they_access(source):
    # a pointer that the compiler has lost sight of (it went through integers or asm) makes flat accesses: LDS counts them
    # too, and what waits for one waits for all LDS reads
    text = compiled(source)[1]
    assert re.search(r"^\s+global_load", text, re.M)
    assert not re.findall(r"^\s+flat_\w+", text, re.M)


def test_inline_assembly_declares_the_registers_it_names():
    # m0, vcc and the like, written inside a block and not among its clobbers, would be lost to a compiler that keeps a value there
    blocks = 0
    for name in sorted(os.listdir(build.CSRC)):
        with open(os.path.join(build.CSRC, name)) as f:
            text = f.read()
        for stmt in re.findall(r"\basm(?:\s+volatile)?\s*\((.*?)\);", text, re.S):
            parts = re.split(r":(?=(?:[^\"]*\"[^\"]*\")*[^\"]*$)", stmt)  # at the colons outside of strings
            clobbers = parts[3] if len(parts) > 3 else ""
            for line in re.split(r"\\n\\t|\\n", "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', parts[0]))):
                written = re.match(r"\s*[sv]_\w+\s+(m0|vcc\w*|exec\w*|scc)\b", line)
                blocks += 1
                assert not written or '"%s"' % written.group(1) in clobbers, (name, line)
    assert blocks > 10
