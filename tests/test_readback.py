"""The read-back of grid arrays (rhybrid_amd/csrc/rh_readback.hpp) gives what a
plain loop gives, value for value, and passes on the error of a copy that fails:
tests/readback_check.cpp compiled on the host (no GPU)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_readback_matches_plain_loop(tmp_path):
    exe = str(tmp_path / "readback_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-o", exe, os.path.join(HERE, "readback_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
