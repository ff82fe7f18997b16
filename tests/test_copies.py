"""Copies between device ranges and the caller's arrays on the host, with and
without pinned memory and threads, tests/copy_check.cpp."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_copies_without_pinned_memory_or_threads(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = tmp_path / "copy_check"
    build = subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                            "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"),
                            os.path.join(ROOT, "tests", "copy_check.cpp"), "-o", str(exe), "-lpthread", "-ldl"],
                           capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout
