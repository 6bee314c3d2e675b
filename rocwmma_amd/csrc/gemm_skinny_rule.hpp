// Which problems the weight-streaming kernels of gemm_skinny.hip take (A row-major, B col-major, C / D row-major, 32-bit results).  Plain
// C++, so that the choice can be looked at on the host.
#ifndef ROCWMMA_AMD_CSRC_GEMM_SKINNY_RULE_HPP
#define ROCWMMA_AMD_CSRC_GEMM_SKINNY_RULE_HPP

#include <cstdint>

namespace rocwmma_amd
{
    constexpr uint32_t kSkinnySlices = 4;   // K slices per block of weight rows
    constexpr uint32_t kSkinnyKBytes = 128; // bytes of K per fragment step (128 8-bit or 64 16-bit elements)
    constexpr uint32_t kSkinnyMaxA   = 131072; // bytes of LDS the token matrix may take
    constexpr uint32_t kSlicedWaves  = 8;
    constexpr uint32_t kSlicedNB     = 2; // blocks of 16 weight rows per wave
    constexpr uint32_t kSlicedCols   = kSlicedWaves * kSlicedNB * 16u; // output columns per workgroup of the K-sliced kernel

    // 16 or 32 rows, all of A in LDS
    constexpr bool skinnyHoldsA(uint32_t m, uint64_t kBytes)
    {
        return m <= 32u && m * kBytes <= kSkinnyMaxA;
    }

    // K steps of a wave's slice that the kernel with all of A in LDS fetches together, as many as divide the slice, up to 8; 0: not its
    // problem.
    constexpr uint32_t skinnySteps(uint32_t m, uint32_t n, uint64_t kBytes, uint32_t units)
    {
        // whole 1 KiB copies per row of A, whole fragment steps per K slice
        if(!skinnyHoldsA(m, kBytes) || m % 16u != 0u || n % 16u != 0u || kBytes % 1024u != 0u)
            return 0u;
        // Up to 32 columns per compute unit the kernel for few rows is faster (gemm_few_rows.hpp; int8, 16 rows, n = 2048, 4096, 8192, K =
        // 4096: 10.3 -> 4.9, 10.4 -> 6.5, 12.2 -> 8.7 us; 32 rows 11.6 -> 5.3, 11.7 -> 6.9, 14.0 -> 8.6), beyond them within 10 % of
        // this one on either side (14336 x 4096 13.6 / 13.1 and 15.6 / 14.4, x 1024 4.9 / 5.3 and 5.6 / 6.2, 28672 x 1024 7.0 / 9.3).
        if(n <= 32u * units)
            return 0u;
        const uint64_t steps = kBytes / (kSkinnySlices * kSkinnyKBytes);
        return steps % 8u == 0u ? 8u : (steps % 4u == 0u ? 4u : 2u);
    }

    // K slices of the K-sliced kernel (16 and 32 rows only when all of A does not fit the LDS); 0: not its problem.
    constexpr uint32_t kSlicesOf(uint32_t m, uint32_t n, uint64_t kBytes, uint32_t computeUnits)
    {
        // (n: the kernel that initialises D counts 4-element groups in 32 bits)
        if(skinnyHoldsA(m, kBytes) || m % 16u != 0u || n % 16u != 0u || n > (1u << 24) || kBytes % 1024u != 0u)
            return 0u;
        // From 64 rows on the blocked kernel is as fast or faster, in one launch and without atomic adds.  Below, K is what decides,
        // alike for 8- and 16-bit types: the blocked kernel has one workgroup walk all of K (about 2.4 us per KiB of it), here
        // the second launch and the atomic adds of every slice (more with more columns) come on top of the weights.  48 rows,
        // n columns, int8, blocked / here in us:
        //     K bytes     n = 256      4096         7168         8192         14336        28672
        //        4096   11.7 / 13.6  11.9 / 14.8  15.0 / 17.5  15.4 / 18.0  17.4 / 22.6  29.7 / 32.6
        //        6144   16.2 / 14.0  19.5 / 16.7  20.9 / 19.8  21.1 / 20.9  23.1 / 32.1  39.0 / 55.6
        //        8192   20.5 / 13.6  25.3 / 18.1  26.5 / 22.5  27.0 / 24.7  31.2 / 32.0  51.8 / 59.6
        //       28672   64.2 / 14.2  81.1 / 32.2  85.6 / 57.4  87.7 / 60.7
        // (float16 with 6144 bytes and n = 7168, 8192: 48 rows 20.8 / 21.1, 21.2 / 22.4; 32 rows, fewer adds, 20.4 / 18.2, 20.6 / 19.3.)
        const uint64_t perUnit   = kBytes / (m > 32u ? 256u : 192u); // columns
        const bool     fewerAdds = n <= computeUnits * (perUnit < 32u ? perUnit : 32u);
        if(m >= 64u || kBytes <= 4096u || !fewerAdds)
            return 0u;
        // whole 1 KiB copies per row and whole batches of fragment steps per slice, the A slice within 128 KiB of LDS; as few slices as
        // fill the compute units
        const uint32_t groups = (n + kSlicedCols - 1u) / kSlicedCols;
        const uint32_t units  = static_cast<uint32_t>(kBytes / 1024u);
        uint32_t       slices = 0;
        for(uint32_t s = 1; s <= units; ++s)
        {
            if(units % s != 0u || m * (kBytes / s) > kSkinnyMaxA)
                continue;
            slices = s;
            if(groups * s >= computeUnits * 3u / 4u)
                break;
        }
        return slices;
    }
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_SKINNY_RULE_HPP
