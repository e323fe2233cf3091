"""The turns of the FP64 ring kernel (gh_turn.h) on CPU threads under ThreadSanitizer: what one
turn writes is ordered before the next turn's reads."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_turns_order_their_writes(tmp_path):
    exe = str(tmp_path / "turn_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread", "-o", exe,
                        os.path.join(ROOT, "tests", "host", "turn_check.cpp")],
                       capture_output=True, text=True)
    if r.returncode != 0 and "tsan" in r.stderr:
        pytest.skip("ThreadSanitizer runtime not available: " + r.stderr[-200:])
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, TSAN_OPTIONS="exitcode=66"))
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer cannot run here: " + r.stderr[-200:])
    assert r.returncode == 0 and r.stdout.strip() == "0 wrong", r.stdout + r.stderr
