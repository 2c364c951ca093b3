"""The single-level Vanka kernels hold their state in registers: a sweep is bound by FP64
issue, and the kernel that loops over tiles once spilled 348 bytes a lane, which made levels
above 2048^2 cells 20 to 37% slower.  This reads the compiler's own resource report for the
library's flags: at most 64 bytes (8 doubles) of spill a lane."""
import os
import re
import subprocess

import pytest

from glide_amd import build

LIMIT = 64


def test_vanka_kernels_do_not_spill(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    flags = [f for f in build.FLAGS if f not in ("-shared",)]
    src = os.path.join(build.CSRC, "glide_hip.hip")
    r = subprocess.run([build.HIPCC, *flags, "-I", os.path.join(build.ROOT, "include"), "-I", build.CSRC,
                        "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-S", "-o", str(tmp_path / "k.s"), src],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    spill = {}
    for block in r.stderr.split("Function Name: ")[1:]:
        name = block.split()[0]
        if re.search(r"k_vanka(_fold|_multi|_rows)?I", name):
            spill[name] = int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", block).group(1))
    assert len(spill) >= 12, sorted(spill)
    over = {k: v for k, v in spill.items() if v > LIMIT}
    assert not over, over
