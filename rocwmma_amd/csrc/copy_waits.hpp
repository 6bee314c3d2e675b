// How many vector-memory operations a wave may have in flight while it waits for direct copies into LDS.  Plain C++, so
// that the counts can be checked on the host.
//
// Copies into LDS complete in the order they were issued among themselves, and only among themselves: loads into
// registers and stores may retire in front of older copies (loads have been seen to, with a cold cache).  A wait that
// counted one of those as in flight would pass with a copy outstanding as soon as it had retired, so only younger copies
// count.  Anything else that is still in flight makes the wait longer, never too short.
#ifndef ROCWMMA_AMD_CSRC_COPY_WAITS_HPP
#define ROCWMMA_AMD_CSRC_COPY_WAITS_HPP

#include <cstdint>

namespace rocwmma_amd
{
    // C staged through `buffers` LDS buffers: `groups` groups of `copies` copies each, the first `buffers` of them issued at once,
    // group g + buffers when group g has been read and its results have been stored.  In flight when group `group` must have
    // landed: the copies of the groups issued behind it.
    constexpr uint32_t stagedCInFlight(uint32_t group, uint32_t groups, uint32_t copies, uint32_t buffers = 2u)
    {
        const uint32_t behind = groups - 1u - group;
        return (behind < buffers - 1u ? behind : buffers - 1u) * copies;
    }
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_COPY_WAITS_HPP
