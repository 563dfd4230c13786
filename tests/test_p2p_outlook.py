"""What a context remembers of its problems' P2P (on the CPU)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_p2p_outlook(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-Wall", "-std=c++17", "-o", exe,
                    os.path.join(HERE, "native", "p2p_outlook_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
