// Limits of a launch.  Plain C++, so that they can be checked on the host.
#ifndef ROCWMMA_AMD_CSRC_LAUNCH_LIMITS_HPP
#define ROCWMMA_AMD_CSRC_LAUNCH_LIMITS_HPP

#include <cstdint>

namespace rocwmma_amd
{
    // A launch counts its threads along a grid dimension in 32 bits: the samples of a batch that one takes, with `perGroup`
    // samples to a workgroup of `threads`.  (27 x 128 float32 samples are the work of four waves each: a batch of 2^24 of them,
    // which fits the memory, is more than one launch.)
    constexpr uint32_t samplesPerLaunch(uint32_t threads, uint32_t perGroup)
    {
        return (0xFFFFFFFFu / threads) * perGroup;
    }

    // f(first sample, samples) for every launch of a batch, in order, until one returns something other than 0.
    template <typename F>
    int forEachLaunch(uint32_t batch, uint32_t threads, uint32_t perGroup, F&& f)
    {
        const uint32_t most = samplesPerLaunch(threads, perGroup);
        for(uint32_t first = 0; first < batch;)
        {
            const uint32_t count = batch - first < most ? batch - first : most;
            if(const int rc = f(first, count))
                return rc;
            first += count;
        }
        return 0;
    }
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_LAUNCH_LIMITS_HPP
