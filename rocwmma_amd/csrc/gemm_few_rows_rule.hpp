// What the kernel for few token rows (gemm_few_rows.hpp) costs, and which of its tiles a problem takes.  Plain C++, so that the
// choice can be checked on the host.
#ifndef ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP
#define ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP

#include <cstdint>

namespace rocwmma_amd
{
    constexpr uint32_t kFewMaxRows = 128u;
    constexpr uint32_t kFewStep    = 128u; // bytes of K per step
    constexpr uint32_t kFewLds     = 163840u;

    // blocks of 16 rows of A that the kernel for m rows has
    constexpr uint32_t fewRowBlocks(uint32_t m)
    {
        const uint32_t blocks = (m + 15u) / 16u;
        return blocks <= 4u ? blocks : (blocks <= 6u ? 6u : 8u);
    }
    constexpr uint32_t fewWaves(uint32_t mb, uint32_t nb)
    {
        return mb + nb <= 3u ? 8u : 4u;
    }
    // steps that a wave has in LDS
    constexpr uint32_t fewRing(uint32_t mb, uint32_t nb)
    {
        return kFewLds / (fewWaves(mb, nb) * (mb + nb) * 16u * kFewStep);
    }
    // (others are never chosen over the blocked kernel: with that many weight rows per workgroup it has enough tiles itself)
    constexpr bool fewHasTile(uint32_t mb, uint32_t nb)
    {
        return nb == 1u || (nb == 2u && mb <= 4u) || (nb == 4u && mb == 1u);
    }

    // Microseconds: a start, the start of each further round of workgroups, and per KB of K what a workgroup's copies take by
    // itself (per round) and more when all compute units copy.  Fitted to 700 timings of all tiles (16 to 128 rows, 1024 to 28672
    // columns, K of 1 to 16 KB, int8, fp8, float16, bfloat16 with GELU; weights from HBM), 10 % off on average.
    struct FewCost
    {
        float alone, shared;
    };
    constexpr FewCost fewCost(uint32_t mb, uint32_t nb)
    {
        constexpr FewCost kCosts[6][3] = {{{0.165f, 0.591f}, {0.307f, 1.02f}, {0.604f, 1.9f}}, {{0.37f, 0.563f}, {0.515f, 1.04f}},
                                          {{0.41f, 0.775f}, {0.707f, 1.16f}},                  {{0.575f, 0.81f}, {1.26f, 0.992f}},
                                          {{1.3f, 0.652f}},                                    {{1.8f, 0.71f}}};
        return kCosts[mb <= 4u ? mb - 1u : (mb == 6u ? 4u : 5u)][nb == 4u ? 2u : nb - 1u];
    }
    constexpr float fewTime(uint32_t m, uint32_t n, float kKB, uint32_t nb, uint32_t units)
    {
        const uint32_t groups = (n + 16u * nb - 1u) / (16u * nb), rounds = (groups + units - 1u) / units;
        const FewCost  c      = fewCost(fewRowBlocks(m), nb);
        return 3.22f + 1.57f * static_cast<float>(rounds - 1u)
               + kKB * (c.alone * static_cast<float>(rounds) + c.shared * static_cast<float>(groups) / static_cast<float>(units));
    }

    struct FewChoice
    {
        uint32_t nb; // blocks of 16 weight rows per workgroup
        float    time;
    };
    // The blocked kernel keeps what it is estimated to do in less than this many times the time here: its estimates (13-20 % off, too
    // low rather than too high where K is long) and these miss by as much.  234 problems of up to 128 rows drawn at random and the fastest of both
    // 0.786 of the blocked kernel's and the weight-streaming kernels' times in the geometric mean; chosen with 1 / 0.9 0.802, one or
    // two slower; with 1 0.800 and seven slower.
    constexpr float kFewMargin = 1.0f / 0.9f;

    constexpr FewChoice cheapestFew(uint32_t m, uint32_t n, uint64_t kBytes, uint32_t units)
    {
        const float kKB  = static_cast<float>(kBytes) * 1e-3f;
        FewChoice   best = {1u, fewTime(m, n, kKB, 1u, units)};
        for(uint32_t nb = 2u; nb <= 4u; nb *= 2u)
            if(fewHasTile(fewRowBlocks(m), nb) && fewTime(m, n, kKB, nb, units) < best.time)
                best = FewChoice{nb, fewTime(m, n, kKB, nb, units)};
        return best;
    }
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_RULE_HPP
