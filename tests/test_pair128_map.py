"""The batched closure's pair passes in 128 x 128 tiles cover the 64 x 64 tasks they stand for
(tests/cpp/pair128_check.cpp, against the library's own plan builder, on the CPU)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pair_tiles_cover_the_tasks(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    libdir = os.path.join(ROOT, "fastapsp_amd", "_lib")
    exe = str(tmp_path / "pair128_check")
    r = subprocess.run([hipcc, "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "pair128_check.cpp"),
                        "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "fastapsp_amd", "csrc"), "-L" + libdir, "-lfap_amd",
                        "-Wl,-rpath," + libdir, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
