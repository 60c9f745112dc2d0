"""Calls whose read-back from the device fails give back what they allocated
(tests/cpp/failed_readback.cpp, which runs the library over a stand-in for the
HIP runtime and needs no GPU)."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_failed_readback():
    cpp = os.path.join(HERE, "cpp")
    exe = os.path.join(cpp, "failed_readback")
    if not os.path.exists(exe):  # (build() compiles it)
        subprocess.run(["make", "-s", "-C", cpp], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "dump: read-back 0 fails, memory given back" in res.stdout
    assert "FAILURES 0" in res.stdout
