// ehp_tile_rules.hpp -- the tiles that 2D launches take by their size.
#pragma once

#include "ehp_joseph_tile.hpp"

#include <algorithm>

namespace ehp
{
    // Tiles of the 2D voxel forward: up to 256 pixels, narrower ones (down to 16, widths evened) until a
    // launch over `poses` poses has four blocks a CU. Blobs, us: 92 x 80 / 70 poses 16: 26.7, 256: 41; 150^2 in
    // FP64 / 150 32: 101, 256: 154; 256^2 / 180 64: 125, 256: 206; 300 x 380 / 524 256: 322, 64: 431.
    inline TileCfg voxel_tile2d(int det, int64_t poses, int cus)
    {
        const int64_t most = (det + 15) / 16, want = (4 * (int64_t) cus + poses - 1) / poses;
        const int nt = (int) std::max<int64_t>((det + 255) / 256, std::min(most, want));
        return TileCfg{(det + nt - 1) / nt, 1, 1};
    }

    // Tiles of the 2D Joseph back projection for a launch over nvox voxels (one problem's, or all of a batch's) on
    // a device of cus compute units
    inline TileCfg joseph_tile2d(int64_t nvox, int cus)
    {
        const int t = nvox >= (int64_t) 1024 * cus ? 32 : (nvox >= (int64_t) 256 * cus ? 16 : 8);
        return TileCfg{t, t, 1};
    }

    // The tile of one of a batch's operators: the caller's where tile() chose it, else the rule's for the launch
    // over the whole batch.
    inline TileCfg batch_tile(const TileCfg& own, bool set_by_caller, const TileCfg& whole)
    {
        return set_by_caller ? own : whole;
    }
} // namespace ehp
