"""The sweeps' index schemes, on the host, from the header that the kernels use: tiles dealt
to the XCDs (each once), several sweeps a launch (each cell one owner, stale cells outside
the owned ones) and the updates pending between tiles (inside the scratch, apart)."""
import os
import subprocess

import pytest

from glide_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_index_schemes(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "check")
    subprocess.run([build.HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-I", os.path.join(build.ROOT, "include"),
                    "-I", build.CSRC, "-o", exe, os.path.join(HERE, "tiling", "check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert int(out.stdout.split()[1]) > 1000000
