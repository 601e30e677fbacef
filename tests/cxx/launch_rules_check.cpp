// launch_rules_check.cpp -- the rules that size the back projections' launches, on the CPU.
//
// Built with g++ against the headers that the library's host code uses. Used by tests/test_launch_rules.py.
#include "ehp_joseph_tile.hpp"

#include <algorithm>

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
