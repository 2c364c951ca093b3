"""Tile height -1 gives the JVP and VJP back the choice by level size, which any other
value takes from the process; what lies outside the documented values is refused."""
import os

import pytest

from glide_amd import _lib


def test_choice_by_level_size_can_be_restored():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    for ty in (0, 4, 6, 8, -1):
        _lib.call("glide_set_tile_height", 1, ty)
    for kernel, ty in ((1, -2), (1, 5), (1, 16), (0, -1), (0, 6), (2, 4)):
        with pytest.raises(_lib.GlideError) as e:
            _lib.call("glide_set_tile_height", kernel, ty)
        assert e.value.code == _lib.GLIDE_E_ARG
