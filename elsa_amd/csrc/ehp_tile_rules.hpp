// ehp_tile_rules.hpp -- the tiles and wavefronts that launches take by their size, which of them two axes share, and
// the order of a forward's.
#pragma once

#include "ehp_joseph_tile.hpp"

#include <algorithm>
#include <cmath>

namespace ehp
{
    // Tiles of the 2D voxel forward: up to 256 pixels, narrower ones (down to 16, widths evened) until a
    // launch over `poses` poses has four blocks a CU; a detector that fits one tile is left whole from three and a
    // half. Blobs, us: 92 x 80 / 70 poses 16: 26.7, 256: 41; 150^2 in FP64 / 150 32: 101, 256: 154; 256^2 / 180
    // 64: 125, 256: 206; 300 x 380 / 524 256: 322, 64: 431; 128^2 on 190 / 960 190: 84, 95: 90; 64^2 on 95 / 960 95: 31,
    // 48: 38; 128^2 on 190 / 480 95: 55, 190: 69.
    inline TileCfg voxel_tile2d(int det, int64_t poses, int cus)
    {
        if (det <= 256 && 2 * poses >= 7 * (int64_t) cus)
            return TileCfg{det, 1, 1};
        const int64_t most = (det + 15) / 16, want = (4 * (int64_t) cus + poses - 1) / poses;
        const int nt = (int) std::max<int64_t>((det + 255) / 256, std::min(most, want));
        return TileCfg{(det + nt - 1) / nt, 1, 1};
    }

    // Tiles of an operator's 2D Joseph back projection over n0 x n1 voxels on a device of cus compute units: 32 x 32 from
    // one a CU on, where they come out even, that is unless a CU in eight would be idle while the last run. Back
    // projections, us, with 32 / 16 at 361 poses, magnification 1.05 (3): 512^2 (256 tiles) 109 / 123 (428 / 476),
    // 560^2 (324) 195 / 137 (803 / 566), 481 x 673 (352) 203 / 153 (816 / 656), 680^2 (484) 201 / 207 (829 / 848), 724^2 (529)
    // 280 / 219 (992 / 955), 800^2 (625) 315 / 241 (1250 / 1072), 1024^2 (1024) 353 / 357 (1608 / 1673).
    inline TileCfg joseph_tile2d(int n0, int n1, int cus)
    {
        const int64_t nvox = (int64_t) n0 * n1, tiles = (int64_t) ((n0 + 31) / 32) * ((n1 + 31) / 32);
        const int64_t places = (tiles + cus - 1) / cus * cus;
        const bool even = 8 * tiles >= 7 * places;
        const int t = nvox >= (int64_t) 1024 * cus && even ? 32 : (nvox >= (int64_t) 256 * cus ? 16 : 8);
        return TileCfg{t, t, 1};
    }

    // Tiles of a batch's over nvox voxels in all, whose workgroups have 256 threads (an operator's few tiles have 1024):
    // smaller ones for longer, as a CU needs several. Back projections, us, with 8 / 16 / 32: 64 problems of 32^2 /
    // 48 poses (256 voxels a CU) 22 / 31 / 60, 16 of 64^2 / 90 (256) 29 / 40 / 82, 24 of 100^2 / 100 (937) 66 / 50 / 91, 16 of
    // 128^2 / 180 (1024) 109 / 71 / 148 and at magnification 3 304 / 283 / 406, 32 of them (2048) 202 / 125 / 156, 64 (4096)
    // 376 / 200 / 195; 64 of 128^2 .. 512^2 16: 1446, 32: 1129.
    inline TileCfg joseph_batch_tile2d(int64_t nvox, int cus)
    {
        const int t = nvox >= (int64_t) 4096 * cus ? 32 : (nvox >= (int64_t) 512 * cus ? 16 : 8);
        return TileCfg{t, t, 1};
    }

    // la planes of at most w x w voxels, the widths evened over the volume
    inline TileCfg even_tile(const Dims& dims, int la, int w)
    {
        auto even = [&](int n) { return (n + (n + w - 1) / w - 1) / ((n + w - 1) / w); };
        return TileCfg{la, std::max(even(dims.vol[0]), even(dims.vol[1])),
                            std::max(even(dims.vol[1]), even(dims.vol[2]))};
    }

    // Tiles of a launch over two driving axes (the first and the last, as about any axis of rotation)
    inline int64_t two_axis_tiles(const Dims& dims, const TileCfg& tc)
    {
        int64_t n = 0;
        for (int a = 0; a < 3; a += 2) {
            int nA, nB, nC;
            tile_counts(dims, tc, a, nA, nB, nC);
            n += (int64_t) nA * nB * nC;
        }
        return n;
    }

    inline bool two_axes(int axes)
    {
        return axes == 3 || axes == 5 || axes == 6;
    }

    // The driving axes that occur and, of these, the poses with the rarest and the commonest
    struct AxisPoses {
        int axes, least, most;
    };

    inline AxisPoses axis_poses(const int* pose_axes, int n)
    {
        int with[3] = {0, 0, 0};
        AxisPoses r{0, n, 0};
        for (int p = 0; p < n; ++p) {
            r.axes |= pose_axes[p];
            for (int a = 0; a < 3; ++a)
                with[a] += (pose_axes[p] >> a) & 1;
        }
        for (int a = 0; a < 3; ++a) {
            if (!(r.axes & (1 << a)))
                continue;
            r.least = std::min(r.least, with[a]);
            r.most = std::max(r.most, with[a]);
        }
        return r;
    }

    // What the wait for the slowest of a launch's tiles over two driving axes grows with: the samples (Joseph) that a
    // voxel gets, of the poses (pose_axes: their axes) that have the rarer axis, and the spread of the tiles' times, by
    // the rays' density near the source and far off it in the plane of the axes.
    inline double tile_wait(double samples, const Dims& dims, const PoseGeom* poses, const int* pose_axes)
    {
        const AxisPoses with = axis_poses(pose_axes, dims.nposes);
        if (!two_axes(with.axes))
            return 0.0;
        const int rarer = std::min(dims.nposes, 2 * with.least);
        double half2 = 0.0;
        for (int a = 0; a < dims.dim; ++a)
            half2 += with.axes & (1 << a) ? 0.25 * dims.vol[a] * dims.vol[a] : 0.0;
        double spread = 0.0;
        for (int p = 0; p < dims.nposes; ++p) {
            double away2 = 0.0;
            for (int a = 0; a < dims.dim; ++a) {
                const double c = poses[p].C[a] - 0.5 * dims.vol[a];
                away2 += c * c;
            }
            const double away = std::sqrt(away2), half = std::min(std::sqrt(half2), 0.75 * away);
            const double ratio = (away + half) / (away - half);
            spread += ratio * std::sqrt(ratio) / dims.nposes;
        }
        return samples / (double) dims.nvox * rarer / dims.nposes * spread;
    }

    // Whether the tiles of two driving axes run in one launch, over nvox voxels, whose slowest tiles are waited for by
    // `wait` (tile_wait): one launch waits for them once; but both axes' tiles then exchange their sums with the volume
    // by atomics (add_second), about 25 ps a voxel more than reading and writing it. Joseph, us, one launch / two, by
    // poses; m: the magnification, m^2 rays a voxel's face; s: the source's distance in volume sides:
    //   64^3  m1.3 s10     4    29 /  30    48   71 /  93     128^3 m1.05 s100  48   235 /  220    72   293 /  303
    //   96^3  m1.3 s10    12    77 /  76    24  106 / 122     128^3 m1.05 s2    48   (90 degrees)       319 /  413
    //   96^3  m1.05 s100  20    80 /  76    32   95 / 101     128^3 m2 s2       10   251 /  259    20   420 /  467
    //   96^3  m2 s2       10   117 / 154    20  195 / 274     200^3 m2 s3       48   (30 degrees, 2 poses with
    //   128^3 m1.3 s10    24   215 / 194    48  335 / 332                            the rarer axis)   4315 / 4033
    //   256^3 m1.3 s10    24  1265 / 1112   48 2154 / 2142    256^3 m1.05 s100  32  1133 /  863   100  2401 / 2359
    //   256^3 m2 s2       10  1565 / 1634   20 2960 / 3149
    // and Siddon much alike (128^3 m1.3: 24 poses 218 / 212, 48 poses 362 / 372; 2D 1024^2: 12 poses 59 / 48, 24 75 / 76).
    inline bool pair_launch(int axes, int64_t nvox, double wait)
    {
        const double small = 1 << 18, large = 1 << 21, most = 70.0; // 64^3: always, from 128^3 on: most
        return two_axes(axes) && (wait >= most || wait * (large - small) >= most * ((double) nvox - small));
    }

    // Tiles of the smallest launch of a 3D back projection with these driving axes: two run in one launch, one or
    // three in a launch each
    inline int64_t least_launch_tiles(const Dims& dims, const TileCfg& tc, int axes)
    {
        if (two_axes(axes))
            return two_axis_tiles(dims, tc);
        int64_t least = 0;
        for (int a = 0; a < 3; ++a) {
            if (!(axes & (1 << a)))
                continue;
            int nA, nB, nC;
            tile_counts(dims, tc, a, nA, nB, nC);
            const int64_t n = (int64_t) nA * nB * nC;
            least = least == 0 || n < least ? n : least;
        }
        return least;
    }

    // 3D Joseph tiles: eight planes of up to 26 x 26 voxels, the widths evened over the volume (a large
    // cross-section spends less on the halo and on rays that leave sideways); while a launch of two axes has fewer
    // than eight such tiles a CU, four planes of 32 x 32, below three a CU of 24 x 24 and 16 x 16, and
    // below one a CU two planes. Of 32 x 32 four run on a CU at once: up to an eighth more would keep the launch
    // waiting for a few (ms, 4x32x32 / 4x23x23: 79 x 158 x 158, 40 poses at magnification 2, 0.81 / 0.70, 18 poses over 60
    // degrees at 3 1.28 / 1.07). Over a short arc the tiles of one axis have few samples (its poses below 0.7 of the
    // other's) and the launch waits for the other's: twice as many, and more, of these. A launch of one axis: either from 15/16 of four a CU, as four workgroups of
    // 512 threads run on a CU and each launch drains by itself. Back projections, us (512 threads):
    //   two axes
    //   256^3 / 360 poses  8x26x26 8015  4x32x32 7978  8x22x22 8080  8x24x24 8626  8x17x17 8873
    //   the same at magnification 1.05, after a forward each
    //                      8x26x26 6833  4x32x32 7133  8x22x22 6850  8x24x24 7493  8x17x17 7706
    //   192^3 / 270        8x24x24 2558  4x32x32 2715  8x22x22 2839  8x17x17 3045
    //   128^3 / 180        4x32x32  607  8x16x16  613  4x22x22  635  4x16x16  667
    //   96^3 / 120         4x24x24  226  8x16x16  236  4x16x16  243  2x16x16  267
    //   64^3 / 90          4x16x16   81  4x24x24  120  2x16x16  101
    //   three axes, 90 poses
    //   192^3              8x24x24 4777  4x32x32 5030  8x22x22 5125  4x24x24 4839
    //   176^3              8x26x26 4231  4x30x30 4538
    //   160^3              8x23x23 2899  4x32x32 2932  4x23x23 2985  4x16x16 3149
    //   144^3              4x24x24 2395  4x29x29 2744  4x18x18 2211  8x16x16 2311
    //   128^3              4x22x22 1691  4x32x32 1840  4x16x16 1641  8x16x16 1760
    //   112^3              4x16x16 1184  4x28x28 1567  4x23x23 1210  4x19x19 1096
    //   96^3               4x16x16  854  4x24x24 1054  2x24x24  826
    //   short arcs, 48 poses: 30 degrees at magnification 2 from three volume sides, and 50 at 1.05 from a hundred
    //   200^3              8x25x25 3953  4x29x29 3435  4x23x23 3464    8x25x25  619  4x29x29  579  4x23x23  602
    //   160^3              4x32x32 2024  4x23x23 2100  4x16x16 1977    4x32x32  327  4x23x23  332  4x16x16  357
    //   128^3              4x32x32 1506  4x22x22 1270  4x16x16 1125    4x32x32  212  4x22x22  216  4x16x16  201
    //   96^3               4x24x24  734  4x16x16  616  2x16x16  499    4x24x24  133  4x16x16  116  2x16x16  127
    //   one axis, 60 poses
    //   128^3              4x22x22  234  4x32x32  236  4x16x16  214
    //   112^3              4x16x16  170  4x28x28  187  4x19x19  158
    inline TileCfg joseph_tile3d(const Dims& dims, const AxisPoses& with, int cus)
    {
        const int axes = with.axes;
        const bool pair = two_axes(axes), lopsided = pair && 10 * (int64_t) with.least < 7 * (int64_t) with.most;
        const int64_t alone = 15 * (int64_t) cus / 4;
        const int64_t deep = pair ? (lopsided ? 16 : 8) * (int64_t) cus : alone;
        const int64_t enough = pair ? (lopsided ? 8 : 3) * (int64_t) cus : alone;
        TileCfg tc = even_tile(dims, 8, 26);
        if (least_launch_tiles(dims, tc, axes) >= deep)
            return tc;
        for (int w = 32; w >= 16; w -= 8) {
            tc = even_tile(dims, 4, w);
            const int64_t tiles = least_launch_tiles(dims, tc, axes);
            const bool spill = pair && w == 32 && tiles > 4 * (int64_t) cus && 2 * tiles < 9 * (int64_t) cus;
            if (tiles >= enough && !spill)
                break;
        }
        if (least_launch_tiles(dims, tc, axes) < cus)
            tc.LA = 2;
        return tc;
    }

    // How far the detector's columns are off one volume axis over the trajectory (3D): the largest tangent of a pose's
    // angle to the axis nearest to it, 1e30 if that is not the same axis in all. Near 0 the rays of a detector row stay
    // in one slab of the volume.
    inline double trajectory_tilt(const PoseGeom* poses, int n)
    {
        int axis = -1;
        double most = 0.0;
        for (int p = 0; p < n; ++p) {
            const float* v = poses[p].Pinv + 4; // the ray direction's change from row to row
            int k = 0;
            double off = 0.0;
            for (int i = 1; i < 3; ++i)
                k = std::fabs(v[i]) > std::fabs(v[k]) ? i : k;
            for (int i = 0; i < 3; ++i)
                off += i == k ? 0.0 : (double) v[i] * v[i];
            if (!(std::fabs(v[k]) > 0.0f) || (axis >= 0 && k != axis))
                return 1.0e30;
            most = std::max(most, std::sqrt(off) / std::fabs(v[k]));
            axis = k;
        }
        return most;
    }

    // Tile column of block id of a forward launch with tiles_u tiles across, in row bp = id / tiles_u of them. An XCD
    // hands its blocks to its four shader engines in turn, so with an even number of columns an engine would
    // always take the same ones: those past the volume's shadow or the detector's edge would leave it idle. From
    // row to row (every second, where the number is not a multiple of four) the columns turn by one, which
    // gives every engine each column as often. Three 96^3 volumes, 198 x 110 pixels (four tiles of 64, the last
    // nearly empty), 72 poses: 317 -> 206 us; Siddon, 96^3, three driving axes: 797 -> 508.
    EHP_HD inline int turned_column(int64_t id, int64_t bp, int tiles_u)
    {
        const int64_t turn = tiles_u & 1 ? 0 : (tiles_u & 2 ? bp >> 1 : bp);
        return (int) ((id - bp * tiles_u + turn) % tiles_u);
    }

    // Wavefront width (pixels; 64 in all) of an operator's 3D Joseph forward in a batch, from row-pair views: 16 x 4 as
    // in the operator's own launch, 8 x 8 for volumes below 112 voxels, whose detectors the wider blocks (64 x 4
    // pixels) overlap by up to a third and whose rays differ more across a wavefront. Batches, us, 8 x 8 / 16 x 4:
    // four of 64^3 / 64 poses on 95 x 73 90.6 / 94.4, three of 56^3 / 56 on 134 x 64 54.0 / 59.8, three of 72^3 / 48
    // at magnification 2 183 / 200, three of 96^3 / 72 195 / 198, three of 100^3 / 64 at magnification 2 499 / 515,
    // two of 112^3 / 48 153 / 143, three of 160^3 / 72 843 / 742.
    inline int batch_wave_width(const Dims& dims)
    {
        return std::max({dims.vol[0], dims.vol[1], dims.vol[2]}) < 112 ? 8 : 16;
    }

    // The tile of one of a batch's operators: the caller's where tile() chose it, else the rule's for the launch
    // over the whole batch.
    inline TileCfg batch_tile(const TileCfg& own, bool set_by_caller, const TileCfg& whole)
    {
        return set_by_caller ? own : whole;
    }
} // namespace ehp
