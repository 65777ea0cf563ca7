"""The ADMM runner's build when memory runs out, on the CPU (no GPU needed):
tests/runner_build_check.hip refuses each allocation of the build in turn (see
its header).  Setup must not fail for it."""
import os
import subprocess

import pytest

from osqp_amd import build as B

from .conftest import ROOT


def test_refused_allocations_leave_the_runner_off(tmp_path):
    if not os.path.exists(B.HIPCC):
        pytest.skip("needs hipcc")
    exe = tmp_path / "check"
    subprocess.run([B.HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Wno-unused-result", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "osqp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "runner_build_check.hip"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True,
                       env=dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1"))
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
    assert "not asked for, 64 bits, one 1: 0 allocations" in r.stdout
    assert "past the most entries, 64 bits, one 0: 0 allocations" in r.stdout
