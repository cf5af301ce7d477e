"""The broadcast FP64 M2L's host tables under AddressSanitizer + UndefinedBehaviorSanitizer.

tables.cpp is compiled with g++ -fsanitize=address,undefined together with
tests/sanitize/bcast_checks.cpp, which builds the operators of p = 1..16 in the
parts that the kernels run; any sanitizer report or failed check fails the test.
CPU only: no device code is built.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "simplefmm_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_bcast_operators_clean_under_asan_ubsan(tmp_path):
    exe = str(tmp_path / "bcast_checks")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-fno-omit-frame-pointer", os.path.join(HERE, "sanitize", "bcast_checks.cpp"),
                    os.path.join(CSRC, "tables.cpp"), "-o", exe], check=True, capture_output=True, text=True, timeout=300)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)
    out = r.stdout + r.stderr
    assert r.returncode == 0, out[-4000:]
    assert "AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    assert "ok (0 failed checks)" in r.stdout
