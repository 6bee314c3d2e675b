// What the kernel whose waves share K (gemm_few_rows.hpp) costs, and which of its tiles a problem takes.  Plain C++, so that the
// choice can be checked on the host.
#ifndef ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP
#define ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP

#include <cstdint>

namespace rocwmma_amd
{
    constexpr uint32_t kFewStep = 128u; // bytes of K per step
    constexpr uint32_t kFewLds  = 163840u;

    constexpr uint32_t fewWaves(uint32_t mb, uint32_t nb)
    {
        return mb + nb <= 3u ? 8u : 4u;
    }
    // steps that a wave has in LDS
    constexpr uint32_t fewRing(uint32_t mb, uint32_t nb)
    {
        return kFewLds / (fewWaves(mb, nb) * (mb + nb) * 16u * kFewStep);
    }

    // Tiles: mb blocks of 16 rows of A against nb blocks of 16 weight rows.  Microseconds per KB of K: what a workgroup's copies take by
    // themselves (per round of workgroups), and more when all compute units copy.  With a start and the start of each further round
    // fitted to 700 timings (16 to 128 rows, 1024 to 28672 columns, K of 1 to 16 KB, int8, fp8, float16, bfloat16 with GELU; weights
    // from HBM), 10 % off on average.  (Tiles of 6 and 8 blocks of A, and of 4 weight blocks against several of A, were never the
    // fastest way.)
    struct FewCost
    {
        uint32_t mb, nb;
        float    alone, shared;
    };
    constexpr uint32_t kFewTiles            = 9;
    constexpr FewCost  kFewCosts[kFewTiles] = {{1, 1, 0.165f, 0.591f}, {1, 2, 0.307f, 1.02f}, {1, 4, 0.604f, 1.9f},
                                               {2, 1, 0.37f, 0.563f},  {2, 2, 0.515f, 1.04f}, {3, 1, 0.41f, 0.775f},
                                               {3, 2, 0.707f, 1.16f},  {4, 1, 0.575f, 0.81f}, {4, 2, 1.26f, 0.992f}};

    struct FewChoice
    {
        uint32_t mb, nb;
        float    time;
    };
    // (All in 32 bits and without a division per tile but one: a small call's host time is what this is part of.)
    constexpr FewChoice cheapestFew(uint32_t m, uint32_t n, uint64_t kBytes, uint32_t units)
    {
        const uint32_t rows = m / 16u, cols = n / 16u; // blocks
        FewChoice      best = {0u, 0u, 1e30f};
        // (more than any tile here is good for; K of one step, which no two waves share: the blocked kernel was estimated faster for every m and n)
        if(static_cast<uint64_t>(rows) * cols > 12u * units || kBytes <= kFewStep)
            return best;
        const uint32_t by[4] = {rows, (rows + 1u) / 2u, (rows + 2u) / 3u, (rows + 3u) / 4u};
        const float    kKB = static_cast<float>(kBytes) * 1e-3f, perUnit = 1.0f / static_cast<float>(units);
        for(FewCost const& c : kFewCosts)
        {
            // (workgroups of several blocks of rows are dealt out over the XCDs by their weights: eight columns of workgroups at a time)
            const uint32_t groupsM = by[c.mb - 1u], groupsN = (cols + c.nb - 1u) >> (c.nb >> 1);
            const uint32_t groups  = groupsM == 1u ? groupsN : groupsM * ((groupsN + 7u) & ~7u);
            const float    rounds  = static_cast<float>((groups + units - 1u) / units);
            const float    time    = 3.22f + 1.57f * (rounds - 1.0f) + kKB * (c.alone * rounds + c.shared * static_cast<float>(groups) * perUnit);
            if(time < best.time)
                best = FewChoice{c.mb, c.nb, time};
        }
        return best;
    }

    // The blocked kernel keeps what it is estimated to do in less than this many times the time here: its estimates (13-20 % off, too
    // low rather than too high where K is long) and these miss by as much.  234 problems of up to 128 rows drawn at random and the fastest
    // of both 0.786 of the blocked kernel's and the weight-streaming kernels' times in the geometric mean; chosen with 1 / 0.9 0.802,
    // one or two slower; with 1 0.800 and seven slower.
    constexpr float kFewMargin = 1.0f / 0.9f;
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP
