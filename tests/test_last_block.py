"""The count by which a launch finds its last block (CPU, the function that the HIP kernels call) is right
again after launches that overlapped."""
import ctypes
import os

import pytest

from test_tile_logic import ROOT, SFX, _build

SRC = os.path.join(ROOT, "tests", "cxx", "last_block_check.cpp")
OUT = os.path.join(ROOT, "tests", "cxx", "_build", f"liblast_block{SFX}.so")


@pytest.fixture(scope="module")
def lib():
    _build(SRC, OUT)
    return ctypes.CDLL(OUT)


@pytest.mark.parametrize("launches", [1, 2, 3, 7])
@pytest.mark.parametrize("blocks", [2, 5, 16, 256])
def test_overlapping_launches_leave_the_count_right(lib, blocks, launches):
    assert lib.last_block(0, blocks, launches, 200) == 0


def test_a_store_of_zero_would_not(lib):
    """The model tells a count that its last block clears with a store from one that wraps."""
    assert lib.last_block(1, 5, 1, 200) == 0
    assert lib.last_block(1, 5, 2, 200) > 20
