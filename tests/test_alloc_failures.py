"""Allocation failures of the generic engine, its programs and the block pool,
checked without a device: a small program built against the headers with the
runtime's allocation calls replaced.  CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_engine_and_programs_report_failed_allocations(tmp_path):
    exe = tmp_path / "check"
    r = subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Wno-everything", "-Xclang", "-target-feature",
                        "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "gpugraph_amd", "csrc"), "-I",
                        os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "program_alloc_check.hip"),
                        "-o", str(exe)], capture_output=True, text=True, timeout=280)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout[-3000:] + r.stderr[-1000:]


def test_block_pool(tmp_path):
    """Reuse, bounds, eviction of the oldest, return on demand and when memory
    is short, several threads, on a host-side device of limited memory."""
    exe = tmp_path / "check"
    native = os.path.join(ROOT, "tests", "native")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(native, "fake_hip"), "-I",
                        os.path.join(ROOT, "gpugraph_amd", "csrc"), os.path.join(native, "pool_check.cpp"), "-o", str(exe),
                        "-lpthread"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout[-3000:]
