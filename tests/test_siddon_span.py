"""The plane-by-plane Siddon forward and the tiles of the back projection against the whole traversal,
bit for bit (CPU, the functions the HIP kernels call): random rays and rays that meet edges, corners and faces exactly (ties), drive
along every axis both ways, at 45 degrees (two crossings of one axis on a plane), and along
faces; voxels off the ray hold NaN, so a read of one shows."""
import ctypes
import os

import numpy as np
import pytest

from test_tile_logic import ROOT, SFX, _build

SRC = os.path.join(ROOT, "tests", "cxx", "siddon_span_check.cpp")
OUT = os.path.join(ROOT, "tests", "cxx", "_build", f"libsiddon_span{SFX}.so")


@pytest.fixture(scope="module")
def lib():
    _build(SRC, OUT)
    return ctypes.CDLL(OUT)


def _rays(dim, vol, rng):
    o, d = [], []
    size = np.array(vol, float)
    for far in (30.0, 3000.0):  # through random points from near and far sources
        for _ in range(150):
            v = rng.standard_normal(dim)
            v /= np.linalg.norm(v)
            o.append(rng.uniform(0, size) - far * v)
            d.append(v)
    steps = np.array(np.meshgrid(*[[-1, 0, 1]] * dim)).reshape(dim, -1).T
    for s in steps:  # diagonals and axes through integer and half-integer points
        if not s.any():
            continue
        for _ in range(6):
            p = rng.integers(0, np.array(vol) + 1) + rng.choice([0.0, 0.5])
            o.append(p - 16.0 * s)
            d.append(s / np.linalg.norm(s))
            o.append(p - 16.0 * s + rng.uniform(-1e-3, 1e-3, dim))  # close to 45 degrees
            d.append(s / np.linalg.norm(s) + rng.uniform(-1e-7, 1e-7, dim))
    od = np.zeros((len(o), 6), np.float32)
    od[:, :dim], od[:, 3:3 + dim] = np.array(o), np.array(d)
    return od


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("vol", [(9, 7, 11), (1, 5, 4), (16, 16, 16), (12, 17), (1, 3)], ids=str)
def test_siddon_planes_equal_traversal_bitwise(lib, vol, dtype):
    dim = len(vol)
    rng = np.random.default_rng(11)
    od = _rays(dim, vol, rng)
    x = rng.standard_normal(int(np.prod(vol))).astype(dtype)
    fn = lib.siddon_span32 if dtype == np.float32 else lib.siddon_span64
    axes = np.zeros(3, np.int64)
    rc = fn(dim, np.array(list(vol) + [1] * (3 - dim), np.int64).ctypes.data_as(ctypes.c_void_p),
            od.ctypes.data_as(ctypes.c_void_p), len(od), x.ctypes.data_as(ctypes.c_void_p),
            axes.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, rc
    assert (axes[:dim] > 0).all()
