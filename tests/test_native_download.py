"""The staged host read (StagingRing::download) on the CPU against the HIP API stand-in, under
AddressSanitizer + UndefinedBehaviorSanitizer and under ThreadSanitizer (it hands parts to helper
threads); no GPU."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")
CSRC = os.path.join(ROOT, "orcaml_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_staged_download(tmp_path, sanitizer):
    exe = str(tmp_path / "download_test")
    r = subprocess.run(["g++", "-std=c++17", "-g", "-O1", f"-fsanitize={sanitizer}", "-fno-sanitize-recover=all", "-pthread",
                        "-I", os.path.join(NATIVE, "hip_stub"), "-I", CSRC, os.path.join(CSRC, "runtime_host.cpp"),
                        os.path.join(NATIVE, "download_test.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1", TSAN_OPTIONS="halt_on_error=1"))
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    assert "all checks passed" in r.stdout
