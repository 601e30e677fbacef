// ehp_last_block.hpp -- the block of a launch that finishes last.
#pragma once

#include "ehp_device.hpp"

namespace ehp
{
    // Counts the calling block (one of its threads calls) among the `blocks` of its launch: true for the block that
    // counts last, which may then read what the others wrote before they counted. The count wraps to 0
    // at `blocks` by itself: any number of whole launches of one size leave it at 0, also launches that overlapped
    // on the device (replays of a captured graph, say), whose own results are then undefined. A store of 0 by the
    // last block would drop what an overlapping launch has counted so far, and no later launch would
    // count right again.
    EHP_HD inline bool counts_last(unsigned int* count, unsigned int blocks)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const unsigned int before = atomicInc(count, blocks - 1);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#else
        const unsigned int before = *count;
        *count = before >= blocks - 1 ? 0 : before + 1;
#endif
        return before == blocks - 1;
    }
} // namespace ehp
