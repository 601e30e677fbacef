// launch_rules_check.cpp -- the rules that size the back projections' launches, on the CPU.
//
// Built with g++ against the headers that the library's host code uses. Used by tests/test_launch_rules.py.
#include "ehp_tile_rules.hpp"
#include "ehp_voxel.hpp"

#include <algorithm>
#include <vector>

using namespace ehp;

// Poses per step of a 2D back projection
extern "C" int steps_2d(int det, int poses, int batch)
{
    Dims d{};
    d.dim = 2;
    d.det[0] = det;
    d.nposes = poses;
    return steps2d(d, batch);
}

// Most LDS of a 2D workgroup over the tiles up to la x tb
extern "C" int64_t most_lds_2d(int la, int tb)
{
    size_t most = 0;
    for (int a = 1; a <= la; ++a)
        for (int b = 1; b <= tb; ++b)
            most = std::max(most, lds2d(tile2d(TileCfg{a, b, 1}), kPoses2d));
    return (int64_t) most;
}

// Tiles of 3D back projections that a device with `limit` bytes of LDS per workgroup took with rows as
// long as the voxels need, and does not take with the rows that they have.
extern "C" int refused_tiles_3d(int64_t limit)
{
    int refused = 0;
    for (int la = 1; la <= 40; ++la)
        for (int tb = 1; tb <= 150; ++tb)
            for (int c = 1; c <= 150; ++c) {
                const TileCfg t{la, tb, c};
                const int64_t rest = (int64_t) batch_lds_bytes(kMaxPoseBatch), rows = (int64_t) la * (c + 2) * 8;
                const int slots = tile_row_slots(3, t);
                if (slots != tb + 2 && slots != ((tb + 2) | 1))
                    return -1;
                refused += rows * (tb + 2) + rest <= limit && rows * slots + rest > limit;
            }
    return refused;
}

// Side of the 2D Joseph tile of an n x n problem in a batch of `total` voxels: its own default tile, left
// alone (0) or chosen by the caller (1)
extern "C" int batch_tile_2d(int n, int64_t total, int set_by_caller)
{
    const int cus = 256;
    const TileCfg own = joseph_tile2d(n, n, cus);
    return batch_tile(own, set_by_caller != 0, joseph_batch_tile2d(total, cus)).LA;
}

// Side of the tiles of a 2D Joseph back projection over n0 x n1 voxels
extern "C" int joseph_tile_2d(int n0, int n1)
{
    return joseph_tile2d(n0, n1, 256).LA;
}

// Columns of the kernel for two voxel projectors in one batch: supports, least and largest scalings, table
// entries; alone: of the first's own kernel (0: the general one)
extern "C" int common_columns(const double* support, const double* smin, const double* smax, const int* n_lut,
                              int* alone)
{
    ColumnNeeds c[2];
    for (int j = 0; j < 2; ++j) {
        const int cols = footprint_cols(support[j], smax[j]);
        c[j] = ColumnNeeds{cols <= kVoxMaxCols ? cols : 0, n_lut[j], support[j], smin[j]};
        if (c[j].cols > 0)
            alone[j] = kernel_cols(cols);
    }
    return common_cols(c, 2);
}

// Whether the columns of `rows` rows of tiles are each taken once, and the most by which the four shader
// engines' blocks of one column differ in number over the rows (-1: not each taken once)
extern "C" int column_spread(int tiles_u, int rows)
{
    std::vector<int> seen((size_t) tiles_u * rows, 0), engine((size_t) tiles_u * 4, 0);
    for (int64_t id = 0; id < (int64_t) tiles_u * rows; ++id) {
        const int c = turned_column(id, id / tiles_u, tiles_u);
        if (c < 0 || c >= tiles_u || seen[(id / tiles_u) * tiles_u + c]++)
            return -1;
        ++engine[c * 4 + id % 4];
    }
    int most = 0;
    for (int c = 0; c < tiles_u; ++c) {
        const auto e = std::minmax_element(&engine[c * 4], &engine[c * 4] + 4);
        most = std::max(most, *e.second - *e.first);
    }
    return most;
}

// Wavefront width of a batch's 3D Joseph forward over x x y x z voxels
extern "C" int wave_width(int x, int y, int z)
{
    Dims d{};
    d.dim = 3;
    d.vol[0] = x;
    d.vol[1] = y;
    d.vol[2] = z;
    return batch_wave_width(d);
}

// The longest view row for four samples at once over n poses with the inverse projections pinv (3D, column-major 4 x 3)
extern "C" int four_samples_up_to(int n, const float* pinv)
{
    std::vector<PoseGeom> g(n);
    for (int p = 0; p < n; ++p)
        std::copy(pinv + 12 * p, pinv + 12 * p + 12, g[p].Pinv);
    return (int) four_sample_row(trajectory_tilt(g.data(), n));
}

// The 3D Joseph back projection's tile of an n^3 volume, as la * 1000 + width, on 256 compute units
extern "C" int joseph_tile(int n, int axes)
{
    Dims d{};
    d.dim = 3;
    d.vol[0] = d.vol[1] = d.vol[2] = n;
    const TileCfg t = joseph_tile3d(d, AxisPoses{axes, 9, 9}, 256);
    return t.TB == t.TC ? t.LA * 1000 + t.TB : -1;
}

// The same of n0 x n1 x n2 voxels with the driving axes 0 and 2, the first in `rare` of 100 poses
extern "C" int tile_3d_box(int n0, int n1, int n2, int rare)
{
    Dims d{};
    d.dim = 3;
    d.vol[0] = n0;
    d.vol[1] = n1;
    d.vol[2] = n2;
    std::vector<int> of(100, 4);
    std::fill(of.begin(), of.begin() + rare, 5);
    const TileCfg t = joseph_tile3d(d, axis_poses(of.data(), 100), 256);
    return (t.LA * 100 + t.TB) * 100 + t.TC;
}

// Parts of the voxel gather's sums and the wavefronts that share them, as parts * 100 + waves
extern "C" int gather_split(int dim, int64_t nvox, int poses, int width, int f64)
{
    Dims d{};
    d.dim = dim;
    d.nvox = nvox;
    d.nposes = poses;
    return gather_part_count(d) * 100 + gather_waves(d, width, f64 != 0);
}

// Width of the 2D voxel forward's tiles on 256 compute units
extern "C" int voxel_tile(int det, int64_t poses)
{
    return voxel_tile2d(det, poses, 256).LA;
}

// Whether the back projection of an n^3 volume runs the tiles of these driving axes in one launch; rays: samples that a
// voxel gets from a pose; away: the source's distance in volume sides; rare: poses with the lowest of the axes
extern "C" int one_launch(int axes, int n, double rays, int poses, double away, int rare)
{
    Dims dims{};
    dims.dim = 3;
    dims.vol[0] = dims.vol[1] = dims.vol[2] = n;
    dims.nposes = poses;
    dims.nvox = (int64_t) n * n * n;
    std::vector<PoseGeom> g(poses);
    std::vector<int> of(poses, axes);
    for (int p = 0; p < poses; ++p) {
        for (int a = 0; a < 3; ++a)
            g[p].C[a] = 0.5f * n + (a == 0 ? (float) away * n : 0.0f);
        if (p >= rare)
            of[p] = axes & (axes - 1);
    }
    return pair_launch(axes, dims.nvox, tile_wait(rays * dims.nvox * poses, dims, g.data(), of.data()));
}
