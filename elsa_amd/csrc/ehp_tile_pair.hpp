// ehp_tile_pair.hpp -- the tiles of two driving axes in one launch (tiled back projections).
#pragma once

#include "ehp_kernels.hpp"
#include "ehp_tile_rules.hpp"

#include <type_traits>

namespace ehp
{
    // Adds v to a voxel that starts at 0 and gets two sums in all, from workgroups in any order: whichever
    // comes second finds the first's sum in exchange for its own and stores both, so the result is the
    // two sums' rounded sum either way.
    template <class T>
    __device__ __forceinline__ void add_second(T* p, T v)
    {
        const T first = __hip_atomic_exchange(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (first != T(0))
            __hip_atomic_store(p, first + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // One driving axis' tiles: the counts along A and b1, of all, and per XCD
    struct TileCounts {
        int nA, nB, n, per_xcd;
    };

    inline TileCounts axis_tiles(const Dims& dims, const TileCfg& tc, int a)
    {
        TileCounts c;
        int nC;
        tile_counts(dims, tc, a, c.nA, c.nB, nC);
        c.n = c.nA * c.nB * nC;
        c.per_xcd = (c.n + 7) / 8;
        return c;
    }

    template <class Job>
    struct BatchTiles { // one driving axis' tiles of a batch
        const Job* jobs;
        const int* block_job;
        int64_t total;
        int per_xcd;
    };

    // fn(first, second) of two of three axes, as constants
    template <class Fn>
    void with_axis_pair(int axes, Fn fn)
    {
        using std::integral_constant;
        if (axes == 3)
            fn(integral_constant<int, 0>{}, integral_constant<int, 1>{});
        else if (axes == 5)
            fn(integral_constant<int, 0>{}, integral_constant<int, 2>{});
        else
            fn(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    }
} // namespace ehp
