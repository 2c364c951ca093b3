"""The sweeps' Newton iteration (newton_device.h) drops factors of two, equal
matrix entries and range handling from the general assembly and LU
(vanka_device.h) without changing a bit.  This runs both on the host over
edge, corner and interior cells, grounded, floating and thickness-limited
states and both grounding-derivative modes, and compares the iterates exactly;
the short exp, log, pow and sigmoid are compared over their whole ranges.
Exact equality is the claim, so there is no tolerance."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_newton_step_equals_the_general_assembly(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "check"
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text("// host build: no HIP runtime needed\n")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", str(tmp_path),
                    "-I", os.path.join(ROOT, "glide_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-o", str(exe),
                    os.path.join(HERE, "newton", "check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ")
    assert int(out.stdout.split()[1]) > 10000
