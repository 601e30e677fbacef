// last_block_check.cpp -- the count that finds a launch's last block, over interleaved launches, on the CPU.
//
// Built with g++ against elsa_amd/csrc/ehp_last_block.hpp (counts_last, the function the HIP kernels
// call). Launches of one size whose blocks run in a random order, one step of one block after the other;
// then a launch by itself, of which only the last block may be told so. Used by tests/test_last_block.py.
#include "ehp_last_block.hpp"

#include <algorithm>
#include <random>
#include <vector>

using namespace ehp;

namespace
{
    // 0: counts_last. 1: an increment, and in a later step of the last block a store of 0.
    int run(int form, int blocks, int launches, unsigned seed)
    {
        std::mt19937 gen(seed);
        unsigned int count = 0;
        int lasts = 0;
        std::vector<bool> reset; // per waiting step: whether it is a block's second step
        reset.assign((size_t) blocks * launches, false);
        auto step = [&](bool second) { // whether the block has another step
            if (second) {
                count = 0;
                return false;
            }
            const bool last = form == 0 ? counts_last(&count, (unsigned) blocks) : count++ == (unsigned) blocks - 1;
            lasts += last;
            return form == 1 && last;
        };
        while (!reset.empty()) {
            const size_t k = gen() % reset.size();
            const bool more = step(reset[k]);
            if (more)
                reset[k] = true;
            else
                reset.erase(reset.begin() + (long) k);
        }
        if (form == 0 && (count != 0 || lasts != launches))
            return 1;
        for (int b = 0; b < blocks; ++b) {
            lasts = 0;
            const bool second = step(false);
            if (second)
                step(true);
            if (lasts != (b == blocks - 1 ? 1 : 0))
                return 2;
        }
        return 0;
    }
} // namespace

// The number of interleavings (of `tries`) after which a launch by itself finds its last block wrongly
extern "C" int last_block(int form, int blocks, int launches, int tries)
{
    int wrong = 0;
    for (int t = 0; t < tries; ++t)
        wrong += run(form, blocks, launches, (unsigned) t) != 0;
    return wrong;
}
