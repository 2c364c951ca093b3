import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) to run")
    config.addinivalue_line("markers", "slow: long-running CPU test")


@pytest.fixture(autouse=True)
def _default_launch_shapes():
    """The library's launch shapes are process-wide: whatever a test and its fixtures leave
    set, the next test starts from the defaults (this is set up first, so it ends last)."""
    yield
    lib = sys.modules.get("glide_amd._lib")
    if lib is None or not os.path.exists(lib.LIB_PATH):
        return
    for kernel in (0, 1):
        lib.call("glide_set_persistence", kernel, 64)
    lib.call("glide_set_tile_height", 0, 0)
    lib.call("glide_set_tile_height", 1, -1)
    lib.call("glide_set_small_levels", 208 * 208, 2)
