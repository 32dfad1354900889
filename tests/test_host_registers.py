"""Registers of the decode kernels, as the compiler reports them: a step kernel that spills pays for it on every page
it walks.  No device is needed."""
import os
import re
import shutil
import subprocess

import pytest

from breccia_amd import build


def test_step_kernels_do_not_spill():
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    proc = subprocess.run([hipcc] + build.HIP_FLAGS + ["--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                          "-I", os.path.join(build.HERE, "..", "include"), "-c", os.path.join(build.CSRC, "decode_attn_mfma.hip"),
                          "-o", os.devnull], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    scratch = dict(re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", proc.stderr, re.S))
    # <STEP, ...>: the template's first argument
    steps = {k: int(v) for k, v in scratch.items() if re.search(r"decode_attn_mfma\w*_kernelILb1E", k)}
    assert len(steps) == 6, sorted(scratch)
    assert not any(steps.values()), steps
