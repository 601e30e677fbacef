"""The rules that size the back projections' launches (CPU, the functions that the library calls)."""
import ctypes
import os

import numpy as np
import pytest

from backends import OracleBackend
from test_tile_logic import ROOT, SFX, _build

SRC = os.path.join(ROOT, "tests", "cxx", "launch_rules_check.cpp")
OUT = os.path.join(ROOT, "tests", "cxx", "_build", f"liblaunch_rules{SFX}.so")


@pytest.fixture(scope="module")
def lib():
    _build(SRC, OUT)
    L = ctypes.CDLL(OUT)
    L.most_lds_2d.restype = ctypes.c_int64
    return L


@pytest.mark.parametrize("det", [1, 1000, (1 << 21) - 1, 1 << 21, (1 << 22) + 5, (1 << 23) - 1])
@pytest.mark.parametrize("poses,batch", [(1, 1), (37, 32), (100000, 1), (100000, 8), (100000, 32)])
def test_rays_of_a_2d_step_count_in_an_int(lib, det, poses, batch):
    """Up to the widest detector that the tiled back projections take (2^23 - 1), with room for the
    workgroup's strides past the last ray."""
    s = lib.steps_2d(det, poses, batch)
    assert 1 <= s <= min(poses, 16 * batch, 512)
    assert s * det + 4 * 1024 < 2 ** 31
    assert s == min(poses, 16 * batch, 512) or det > (1 << 30) // 512


def test_2d_tiles_fit_64_kb(lib):
    assert lib.most_lds_2d(300, 1300) <= 65536


@pytest.mark.parametrize("limit", [65536, 163840])
def test_row_padding_refuses_no_3d_tile(lib, limit):
    assert lib.refused_tiles_3d(ctypes.c_int64(limit)) == 0


def test_a_tile_that_the_caller_chose_stays_in_a_batch(lib):
    """Also when it equals the tile that the operator would have by itself."""
    total = ctypes.c_int64(64 * 512 * 512)
    assert lib.batch_tile_2d(64, total, 0) == 32
    assert lib.batch_tile_2d(64, total, 1) == 8


@pytest.mark.parametrize("ops,alone,both", [
    # support, least and largest scaling, table entries of each
    (((2.0, 1.04, 1.06, 100), (2.0, 1.04, 1.06, 100)), (5, 5), 5),
    (((2.0, 1.04, 1.06, 100), (1.5, 1.04, 1.06, 100)), (5, 4), 5),
    (((1.5, 1.04, 1.06, 100), (2.0, 1.4, 1.9, 100)), (4, 8), 8),
    (((2.0, 1.04, 1.06, 100), (2.0, 1.5, 2.5, 100)), (5, 0), 0),  # a footprint wider than eight
    (((1.0, 0.9, 1.1, 1000), (2.0, 1.4, 1.9, 100)), (4, 8), 0),  # the first's table would not reach as far
], ids=str)
def test_columns_of_a_batch_of_voxel_projectors(lib, ops, alone, both):
    """Operators of different widths share the widest one's kernel."""
    f = lambda i, c: (c * 2)(*(op[i] for op in ops))
    own = (ctypes.c_int * 2)(0, 0)
    got = lib.common_columns(f(0, ctypes.c_double), f(1, ctypes.c_double), f(2, ctypes.c_double),
                             f(3, ctypes.c_int), own)
    assert tuple(own) == alone and got == both


@pytest.mark.parametrize("tiles", list(range(1, 26)) + [64, 97])
def test_columns_of_a_forward_launch(lib, tiles):
    """Every row takes each of its tiles once, and over many rows the four shader engines take each column
    equally often (up to the rows of an unfinished turn)."""
    rows = 4 * tiles * 30
    assert 0 <= lib.column_spread(tiles, rows) <= 1


@pytest.mark.parametrize("vol,width", [((64, 64, 64), 8), ((1, 1, 1), 8), ((111, 111, 111), 8), ((112, 5, 5), 16),
                                       ((5, 112, 5), 16), ((5, 5, 300), 16)], ids=str)
def test_wavefronts_of_a_batch_of_3d_joseph_forwards(lib, vol, width):
    """Narrow ones for small volumes, which 64-pixel blocks overlap too far."""
    assert lib.wave_width(*vol) == width


@pytest.mark.parametrize("beta,row", [(0.0, 2304), (0.015, 2304), (0.03, 1312), (0.3, 1312), (0.4, 800), (0.8, 800),
                                      (np.pi / 2, 800)])
def test_rows_for_four_samples(lib, beta, row):
    """A circle about y takes four over long rows, also slightly tilted; one tilted further, in turn either way, does
    not, and one whose detector columns turn from axis to axis least."""
    poses = [dict(s2c=400.0, c2d=100.0, gamma=a, beta=beta * np.sin(2.0 * a)) for a in np.linspace(0.0, 6.0, 25)]
    g = OracleBackend().setup((40, 50, 60), (70, 60), poses)
    pinv = np.ascontiguousarray(g.Pinv, np.float32)
    assert pinv.size == 25 * 12
    assert lib.four_samples_up_to(25, pinv.ctypes.data_as(ctypes.POINTER(ctypes.c_float))) == row


@pytest.mark.parametrize("n,two,one", [(256, 8026, 8026), (192, 8024, 8024), (176, 8026, 8026), (160, 4032, 8023), (144, 4029, 4024),
                                       (128, 4032, 4022), (112, 4028, 4016), (96, 4024, 4016), (64, 4016, 4016),
                                       (32, 2016, 2016)])
def test_3d_joseph_tiles(lib, n, two, one):
    """By the tiles of one launch: two driving axes run in one, one or three axes in a launch each."""
    assert all(lib.joseph_tile(n, axes) == two for axes in (3, 5, 6))
    assert all(lib.joseph_tile(n, axes) == one for axes in (1, 2, 4, 7))


@pytest.mark.parametrize("dim,n,poses,width,parts,waves", [
    (3, 64, 60, 5, 2, 2), (3, 64, 60, 8, 2, 2), (3, 64, 60, 9, 2, 1), (3, 64, 60, 25, 2, 1),
    (3, 48, 60, 5, 4, 4), (3, 48, 60, 16, 4, 4), (3, 48, 60, 17, 4, 2), (3, 56, 40, 16, 4, 2), (3, 56, 40, 17, 4, 1),
    (3, 40, 40, 5, 8, 8), (3, 40, 40, 16, 8, 8), (3, 40, 40, 24, 8, 4), (3, 40, 40, 25, 8, 2), (3, 24, 24, 25, 4, 4), (3, 8, 1000, 25, 16, 16), (3, 8, 7, 5, 1, 1),
    (3, 128, 500, 25, 1, 1), (2, 64, 90, 50, 16, 16), (2, 400, 360, 50, 4, 4)])
def test_parts_of_the_voxel_gather(lib, dim, n, poses, width, parts, waves):
    """A sum's parts follow from its size alone; fewer wavefronts share them for wide footprints in 3D, whose
    pixels the caches hold for few poses at once."""
    assert lib.gather_split(dim, ctypes.c_int64(n ** dim), poses, width, 0) == parts * 100 + waves
    assert lib.gather_split(dim, ctypes.c_int64(n ** dim), poses, width, 1) == parts * 101


@pytest.mark.parametrize("det,poses,width", [(190, 960, 190), (95, 960, 95), (256, 896, 256), (190, 895, 95),
                                             (257, 960, 129), (190, 480, 64), (1, 1, 1), (1, 5000, 1), (381, 180, 64),
                                             (763, 360, 255), (300, 5000, 150)])
def test_2d_voxel_forward_tiles(lib, det, poses, width):
    """A detector that fits one tile is left whole while the launch has three and a half blocks a CU."""
    assert lib.voxel_tile(det, ctypes.c_int64(poses)) == width


@pytest.mark.parametrize("n,tile", [((79, 158, 158), 42323), ((96, 184, 100), 42423), ((128, 128, 128), 43232),
                                    ((139, 128, 121), 43232), ((147, 164, 76), 43028), ((96, 96, 96), 42424)])
def test_3d_joseph_tiles_of_boxes(lib, n, tile):
    """A few tiles more than run at once make them smaller."""
    assert lib.tile_3d_box(*n, 70) == lib.tile_3d_box(*n, 100) == tile


@pytest.mark.parametrize("n,tile", [((200, 200, 200), 42929), ((160, 160, 160), 42323), ((128, 128, 128), 42222),
                                    ((96, 96, 96), 41616), ((256, 256, 256), 82626), ((51, 51, 206), 41316)])
def test_3d_joseph_tiles_of_short_arcs(lib, n, tile):
    """Smaller where one axis has few of the poses."""
    assert lib.tile_3d_box(*n, 69) == lib.tile_3d_box(*n, 1) == tile


@pytest.mark.parametrize("n0,n1,side", [(16, 16, 8), (256, 255, 8), (256, 256, 16), (511, 512, 16), (512, 512, 32),
                                        (481, 673, 16), (560, 560, 16), (640, 690, 16), (680, 680, 32), (704, 704, 32),
                                        (724, 724, 16), (800, 800, 16), (1024, 1024, 32), (30, 20000, 16)])
def test_2d_joseph_tiles(lib, n0, n1, side):
    """Large ones only where the compute units get them in equal numbers."""
    assert lib.joseph_tile_2d(n0, n1) == side


@pytest.mark.parametrize("problems,n,side", [(64, 32, 8), (16, 64, 8), (32, 64, 16), (24, 100, 16), (16, 128, 16),
                                             (32, 128, 16), (63, 128, 16), (64, 128, 32), (64, 512, 32)])
def test_2d_joseph_tiles_of_a_batch(lib, problems, n, side):
    """Several tiles a compute unit before they grow."""
    assert lib.batch_tile_2d(n, ctypes.c_int64(problems * n * n), 0) == side


@pytest.mark.parametrize("n,rays,away,few,many", [
    (64, 0.1, 100, 0, 1), (96, 1.0, 100, 20, 32), (96, 1.5, 10, 12, 24), (96, 3.6, 2, 2, 10), (128, 1.0, 100, 48, 100),
    (128, 1.5, 10, 24, 50), (128, 3.6, 2, 5, 9), (128, 1.0, 2, 20, 48), (256, 1.0, 100, 48, 100), (256, 8.0, 3, 4, 9),
    (256, 8.0, 0.2, 0, 1)])
def test_two_axes_in_one_launch(lib, n, rays, away, few, many):
    """From as many poses as pay for the atomics, fewer for denser rays and a nearer source; poses with but one of the
    axes do not count, and one or three axes never share a launch."""
    def one(axes, poses, rare=None):
        return lib.one_launch(axes, n, ctypes.c_double(rays), poses, ctypes.c_double(away), poses if rare is None else rare)

    for axes in (3, 5, 6):
        assert one(axes, many) and one(axes, many, (many + 1) // 2)
        assert few == 0 or not one(axes, few)
        assert few == 0 or not one(axes, many, max(few // 4, 1) if few > 1 else 0)
    for axes in (1, 2, 4, 7):
        assert not one(axes, 1000)
