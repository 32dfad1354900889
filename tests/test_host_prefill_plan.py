"""The cut of chunk attention's page walks (csrc/prefill_plan.hpp) over random batches, walked on the host the way the
kernels walk it: tests/cpp/prefill_plan_test.cpp.  Host code only."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def binary(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "prefill_plan_test")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover",
                    os.path.join(HERE, "cpp", "prefill_plan_test.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("seed", [1, 7, 42])
def test_every_cut_covers_every_page_once_inside_the_workspace(binary, seed):
    r = subprocess.run([binary, str(seed), "30000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
