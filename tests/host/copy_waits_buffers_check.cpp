// copy_waits_check.cpp's sequence with four buffers of C per wave: whenever a group is read, all of its copies must have
// landed, and no wait holds longer than it has to.
#include "../../rocwmma_amd/csrc/copy_waits.hpp"

#include <cstdio>
#include <deque>

int main()
{
    int failures = 0;
    for(uint32_t groups = 4; groups <= 16; ++groups)
        for(uint32_t copies = 1; copies <= 16; ++copies)
        {
            std::deque<uint32_t> inFlight; // group of each copy, oldest first
            auto                 issue = [&](uint32_t group) { inFlight.insert(inFlight.end(), copies, group); };
            for(uint32_t g = 0; g < 4u; ++g)
                issue(g);
            for(uint32_t g = 0; g < groups; ++g)
            {
                while(inFlight.size() > rocwmma_amd::stagedCInFlight(g, groups, copies, 4u))
                    inFlight.pop_front();
                if(!inFlight.empty() && inFlight.front() != g + 1u)
                {
                    std::printf("groups %u copies %u: group %u read with group %u the oldest in flight\n", groups, copies, g, inFlight.front());
                    ++failures;
                }
                if(g + 4u < groups)
                    issue(g + 4u);
            }
            if(!inFlight.empty())
                ++failures;
        }
    if(failures == 0)
        std::printf("copy waits OK\n");
    return failures != 0;
}
