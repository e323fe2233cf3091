"""The FP64 pair factor (gh_pairf64.h, the function the direct-sum kernels run) on the CPU:
bit for bit (1/d)/sqrt(d) in three correctly rounded operations."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_pair_factor_correctly_rounded(tmp_path):
    exe = str(tmp_path / "pair_factor_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "host", "pair_factor_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and " 0 wrong" in r.stdout, r.stdout + r.stderr
