// A batch is cut into launches that together take every sample once, each with fewer than 2^32 threads.
#include "../../rocwmma_amd/csrc/launch_limits.hpp"

#include <cstdio>
#include <initializer_list>

int main()
{
    int failures = 0;
    for(uint32_t threads : {64u, 256u, 512u})
        for(uint32_t perGroup : {1u, 2u, 4u, 8u})
            for(uint32_t batch : {1u, 65536u, 16777214u, 16777215u, 16777216u, 16777217u, 67108863u, 67108864u, 134217731u, 4294967295u})
            {
                uint64_t next = 0;
                int      rc   = rocwmma_amd::forEachLaunch(batch, threads, perGroup, [&](uint32_t first, uint32_t count) {
                    const uint64_t groups = (static_cast<uint64_t>(count) + perGroup - 1u) / perGroup;
                    if(first != next || count == 0u || groups * threads > 0xFFFFFFFFull)
                        ++failures;
                    next = static_cast<uint64_t>(first) + count;
                    return 0;
                });
                if(rc != 0 || next != batch)
                    ++failures;
            }
    // an error ends the batch
    int launches = 0;
    if(rocwmma_amd::forEachLaunch(4294967295u, 512u, 1u, [&](uint32_t, uint32_t) { return ++launches == 2 ? 7 : 0; }) != 7 || launches != 2)
        ++failures;
    std::printf(failures == 0 ? "launch limits OK\n" : "%d failures\n", failures);
    return failures != 0;
}
