"""The pointwise arithmetic of FP64 storage (nested equilibria, closed-form
stages, sums by wavefront; uq_amd/csrc/lbm_point.hpp) against the closed forms
and the reference's stage formulas, on the host: tests/point_check.cpp, built
against the header the kernels include."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_point_arithmetic(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = tmp_path / "point_check"
    build = subprocess.run([HIPCC, "-std=c++17", "-O2", "--offload-arch=gfx950", "-I", os.path.join(ROOT, "include"),
                            os.path.join(ROOT, "tests", "point_check.cpp"), "-o", str(exe)],
                           capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout
