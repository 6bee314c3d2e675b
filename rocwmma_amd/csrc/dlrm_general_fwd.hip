// DLRM dot interaction, float16 forward, for samples that do not fit the LDS (dlrm_general.hip has the other kernels of
// those): Z = F F^T of each sample on the blocked GEMM's main loop (gemm_blocked_core.hpp), both operands the sample's
// feature rows, only the tiles that meet the strict lower triangle, one grid for the whole batch.  The triangle leaves packed:
// a wave's results pass through its part of the LDS, freed by then, and go out as pieces of rows, which are
// contiguous in the packed output at any half.
//
// Against 128 x 128 tiles of four waves on one LDS stage with two barriers: (1024, 1024, 64) 108 -> 91 us (860 TFLOP/s
// multiplied, 750 of them wanted), (512, 1024, 32) 28 -> 21, (250, 1024, 16) 18.7 -> 14.1, (700, 136, 40) 21 -> 18.  Bound by a
// tile's copies (64 flop a byte) and, in a sample of few stages, by its first loads and its results.  256 x 256 tiles
// leave more of the chip idle in the last round and multiply more above the diagonal: 100, 34, 32 and 23 us; they are
// ahead from 4096 rows on (129 against 148 us at (4096, 256, 16)), which nothing here is sized for.
#include "gemm_blocked_launch.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    namespace
    {
        // 128 x 128 tiles, two workgroups per compute unit, as the GEMM's rung of that size
        using FwdTile = BlockedConfig<float16_t, float16_t, float32_t, true, true, 2, 2, 4, 4, 2, 2, 16, true, false, false, 0, true>;

        struct __attribute__((packed, aligned(2))) Piece16
        {
            uint32_t w[4];
        };

        // Z(row, column) of a wave's results into the sample's packed output.
        template <typename Cfg>
        struct PackTriangle
        {
            float16_t* out; // entry (1, 0)
            uint32_t   m;
            static constexpr uint32_t Pitch = Cfg::WaveN * 2u + 16u; // bytes per row in LDS
            static_assert(Cfg::Block == 16u && Cfg::Waves * Cfg::WaveM * Pitch <= Cfg::LdsBytes, "a lane owns four columns of one row; LDS size");

            template <typename Acc>
            ROCWMMA_DEVICE ROCWMMA_INLINE void operator()(Acc const& acc, uint32_t wRow, uint32_t wCol) const
            {
                extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];
                typedef uint32_t u32x2_t __attribute__((ext_vector_type(2), may_alias));
                if(wRow >= m || wCol >= min(wRow + Cfg::WaveM, m) - 1u) // (wave uniform) nothing below the diagonal
                    return;
                const uint32_t lane = threadIdx.x & 63u;
                char*          mine = ldsRaw + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (Cfg::WaveM * Pitch);
#pragma unroll
                for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
#pragma unroll
                    for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                    {
                        float16_t h[4];
#pragma unroll
                        for(uint32_t e = 0; e < 4u; ++e)
                            h[e] = static_cast<float16_t>(acc[bi][bj].x[e]);
                        *reinterpret_cast<u32x2_t*>(mine + (bi * 16u + (lane & 15u)) * Pitch + (bj * 16u + 4u * (lane >> 4)) * 2u) = *reinterpret_cast<u32x2_t*>(h);
                    }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                auto rowStart = [&](uint32_t row) { return out + static_cast<size_t>(row) * (row - (row != 0u)) / 2u; };
                if(wRow >= wCol + Cfg::WaveN) // (wave uniform) all of it below the diagonal: 16-byte pieces
                {
                    constexpr uint32_t PerRow = Cfg::WaveN / 8u;
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::WaveM * PerRow / 64u; ++i)
                    {
                        const uint32_t r = i * (64u / PerRow) + lane / PerRow, c = (lane % PerRow) * 8u;
                        if(wRow + r < m)
                            *reinterpret_cast<Piece16*>(rowStart(wRow + r) + wCol + c) = *reinterpret_cast<const Piece16*>(mine + r * Pitch + c * 2u);
                    }
                }
                else
                {
                    for(uint32_t r = 0; r < Cfg::WaveM; ++r)
                        for(uint32_t c = lane; c < Cfg::WaveN; c += 64u)
                            if(wRow + r < m && wCol + c < wRow + r)
                                rowStart(wRow + r)[wCol + c] = *reinterpret_cast<const float16_t*>(mine + r * Pitch + c * 2u);
                }
            }
        };

        template <typename Cfg>
        __global__ void __launch_bounds__(Cfg::Threads) __attribute__((amdgpu_waves_per_eu(Cfg::WavesPerSimd, Cfg::WavesPerSimd)))
            dlrmFwdTileKernel(const float16_t* input, float16_t* output, uint32_t m, uint32_t k, uint32_t batch, uint32_t tiles)
        {
            // all tiles of a sample on one XCD: its features are fetched into one L2
            const uint32_t slot   = blockIdx.x / kXcds;
            const uint32_t sample = (slot / tiles) * kXcds + blockIdx.x % kXcds, t = slot % tiles;
            if(sample >= batch) // (the whole workgroup)
                return;
            uint32_t I = static_cast<uint32_t>((__builtin_sqrtf(8.0f * static_cast<float>(t) + 1.0f) - 1.0f) * 0.5f);
            while(I * (I + 1u) / 2u > t)
                --I;
            while((I + 1u) * (I + 2u) / 2u <= t)
                ++I;
            const uint32_t   J    = t - I * (I + 1u) / 2u;
            const float16_t* feat = input + static_cast<size_t>(sample) * m * k;
            float16_t*       out  = output + static_cast<size_t>(sample) * (k + m * (m - 1u) / 2u);
            if(t == 0u) // bottom-MLP row: the sample's first feature row
                for(uint32_t e = threadIdx.x; e < k; e += Cfg::Threads)
                    out[e] = feat[e];
            gemmTile<Cfg>(I, J, 0u, stagesOf<Cfg>(k), m, m, k, feat, feat, static_cast<const float16_t*>(nullptr), out, k, k, 0u, 0u, 1.0f, 0.0f,
                          StreamKPart{}, TileExtras{}, PackTriangle<Cfg>{out + k, m});
        }

        template <typename Cfg>
        int launchFwd(const void* input, void* output, uint32_t m, uint32_t k, uint32_t batch, hipStream_t stream)
        {
            const uint32_t side = ceilDiv(m, Cfg::MacroM), tiles = side * (side + 1u) / 2u;
            const uint64_t grid = static_cast<uint64_t>(ceilDiv(batch, kXcds)) * kXcds * tiles;
            // (a stage's copies address their source inside a 2 GiB window from the stage origin)
            if(grid > 0x7FFFFFFFull || static_cast<uint64_t>(k) * 2u * Cfg::MacroM >= 0x7FFF0000ull)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            auto kernel = dlrmFwdTileKernel<Cfg>;
            // more than 64 KiB of dynamic LDS needs an explicit opt-in (idempotent, no allocation)
            if(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(Cfg::LdsBytes))
               != hipSuccess)
                return ROCWMMA_AMD_LAUNCH_FAILED;
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(grid)), dim3(Cfg::Threads), Cfg::LdsBytes, stream, static_cast<const float16_t*>(input),
                               static_cast<float16_t*>(output), m, k, batch, tiles);
            return launchStatus();
        }
    } // namespace

    // k a multiple of 8; ROCWMMA_AMD_UNSUPPORTED_SHAPE where 128 feature rows span more than a copy's window
    int launchDlrmFwdTilesF16(const void* input, void* output, uint32_t m, uint32_t k, uint32_t batch, hipStream_t stream)
    {
        return launchFwd<FwdTile>(input, output, m, k, batch, stream);
    }
} // namespace rocwmma_amd
