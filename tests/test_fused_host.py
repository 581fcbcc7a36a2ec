"""The fused kernels' host-checkable parts (exact.hpp) and host tables
(fused_tables.cpp) at the ends of their ranges, built with g++ under
AddressSanitizer and UndefinedBehaviorSanitizer (tests/native/fused_check.cpp):
every check holds, no report."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "aoa_amd", "csrc")
OUT = os.path.join(HERE, "native", "_build", "fused_check")


def test_fused_host_checks():
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-ffp-contract=off", "-fno-omit-frame-pointer", "-pthread",
                    "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I" + CSRC,
                    os.path.join(HERE, "native", "fused_check.cpp"), os.path.join(CSRC, "params.cpp"), os.path.join(CSRC, "fused_tables.cpp"),
                    "-o", OUT],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([OUT], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1:halt_on_error=1"))
    assert r.returncode == 0 and "0 failure(s)" in r.stdout, r.stdout[-3000:] + r.stderr[-6000:]
