// The epilogue of the blocked GEMM waits for copies of C into LDS with stores of D in between.  Plays its sequence of
// operations with copies that land in order and as late as a wait allows, and stores that retire at once (the worst case
// for a count): whenever a group is read, all of its copies must have landed.
#include "../../rocwmma_amd/csrc/copy_waits.hpp"

#include <cstdio>
#include <deque>

int main()
{
    int failures = 0;
    for(uint32_t groups = 2; groups <= 16; ++groups)
        for(uint32_t copies = 1; copies <= 16; ++copies)
        {
            std::deque<uint32_t> inFlight; // group of each copy, oldest first; stores have retired
            auto                 issue = [&](uint32_t group) {
                for(uint32_t i = 0; i < copies; ++i)
                    inFlight.push_back(group);
            };
            issue(0u);
            issue(1u);
            for(uint32_t g = 0; g < groups; ++g)
            {
                while(inFlight.size() > rocwmma_amd::stagedCInFlight(g, groups, copies))
                    inFlight.pop_front();
                for(uint32_t group : inFlight)
                    if(group <= g)
                    {
                        std::printf("groups %u copies %u: group %u read with a copy of it in flight\n", groups, copies, g);
                        ++failures;
                        break;
                    }
                if(g + 2u < groups)
                    issue(g + 2u);
            }
        }
    if(failures == 0)
        std::printf("copy waits OK\n");
    return failures != 0;
}
