// launch_rules_check.cpp -- the rules that size the back projections' launches, on the CPU.
//
// Built with g++ against the headers that the library's host code uses. Used by tests/test_launch_rules.py.
#include "ehp_joseph_tile.hpp"

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
