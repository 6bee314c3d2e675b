// Blocked GEMM for gfx950, one macro tile per workgroup: dispatch over element types, and the block-scaled
// kernels.  The device side (configuration, LDS pipeline, epilogue) is in gemm_blocked_core.hpp, the kernels and
// launch helpers in gemm_blocked_launch.hpp, the tile ladder in gemm_blocked_ladder.hpp; each element type's rungs
// are a translation unit of their own (gemm_blocked_<type>.hip, with the fused epilogue gemm_fused_<type>.hip).
#include "gemm_blocked_launch.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    namespace
    {
        template <typename InT>
        int launchMx(GemmArgs const& g, TileExtras const& ex, hipStream_t stream)
        {
            // 256 x 256 tiles of 16x16x128 blocks with block scales; the tiles of a last round at most half
            // full run as 256 x 128 half tiles, as in the unscaled kernel
            using Big     = BlockedConfig<InT, float32_t, float32_t, true, true, 4, 2, 4, 8, 2, 2, 16, false, true>;
            using BigHalf = BlockedConfig<InT, float32_t, float32_t, true, true, 4, 2, 4, 4, 2, 2, 16, false, true>;
            const int rc  = launchSplitTail<Big, BigHalf>(g, stream, ex);
            if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                return rc;
            return launchCfg<Big>(g, stream, ex);
        }
    } // namespace

    namespace
    {
        // One round of 128 x 64 tiles, more than a quarter full, with at least 4 KiB of K per row.
        bool mxTakesLineTiles(GemmArgs const& g)
        {
            const uint32_t tiles = ceilDiv(g.m, 128u) * ceilDiv(g.n, 64u);
            return g.k % 128u == 0u && g.k >= 4096u && tiles <= computeUnits() && 4u * tiles > computeUnits();
        }

        // Raw: the scales in the caller's order (MxPacked)
        template <typename InT, bool Raw>
        int launchMxMid(GemmArgs const& g, TileExtras const& ex, hipStream_t stream)
        {
            // 128 x 128 tiles of 32x32x64 blocks with block scales, the last row and column of tiles partly
            // filled: any m, n in multiples of 16
            using Mid = BlockedConfig<InT, float32_t, float32_t, true, true, 2, 2, 2, 2, 2, 2, 32, true, true, false, 0, false, Raw>;
            // at most one 128 x 128 tile per two compute units (few token rows against a wide weight matrix):
            // 128 x 64 tiles put twice as many workgroups to work
            using Narrow = BlockedConfig<InT, float32_t, float32_t, true, true, 2, 2, 2, 1, 2, 3, 32, true, true, false, 0, false, Raw>;
            // mxTakesLineTiles: the tile on the ring of four 128-byte stages (whole-line requests, three stages in flight), as the
            // unscaled types' rung of that name: 128 x 14336 x 4096 31 -> 21 us on scales packed beforehand.
            using NarrowLines = BlockedConfig<InT, float32_t, float32_t, true, true, 2, 2, 2, 1, 4, 1, 32, true, true, false, 128, false, Raw>;
            if(mxTakesLineTiles(g))
            {
                const int rc = launchCfg<NarrowLines>(g, stream, ex);
                if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                    return rc;
            }
            if(2u * ceilDiv(g.m, 128u) * ceilDiv(g.n, 128u) <= computeUnits())
                return launchCfg<Narrow>(g, stream, ex);
            return launchCfg<Mid>(g, stream, ex);
        }
    } // namespace

    bool gemmMxBlockedUsesLargeTile(GemmArgs const& g)
    {
        return g.m % 256u == 0u && g.n % 256u == 0u && 2u * (g.m / 256u) * (g.n / 256u) >= computeUnits();
    }

    int launchGemmMxBlocked(int dtypeIn, GemmArgs const& g, const void* packedA, const void* packedB, hipStream_t stream)
    {
        if(g.layoutC != ROCWMMA_AMD_ROW_MAJOR || g.m % 16u != 0u || g.n % 16u != 0u || g.k % 128u != 0u)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        TileExtras ex{};
        ex.mx = MxPacked{packedA, packedB, (g.k / 128u + 1u) / 2u, 0u, 0u, nullptr, nullptr};
        const bool large = gemmMxBlockedUsesLargeTile(g);
        if(dtypeIn == ROCWMMA_AMD_E4M3)
            return large ? launchMx<float8_t>(g, ex, stream) : launchMxMid<float8_t, false>(g, ex, stream);
        if(dtypeIn == ROCWMMA_AMD_E5M2)
            return large ? launchMx<bfloat8_t>(g, ex, stream) : launchMxMid<bfloat8_t, false>(g, ex, stream);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

    int launchGemmMxBlockedRaw(int dtypeIn, GemmArgs const& g, MxScales const& s, void* packedA, void* packedB, hipStream_t stream)
    {
        const bool dwords = ((reinterpret_cast<uintptr_t>(s.a) | reinterpret_cast<uintptr_t>(s.b)) & 3u) == 0u && (s.lda | s.ldb) % 4u == 0u;
        if(g.layoutC != ROCWMMA_AMD_ROW_MAJOR || g.m % 16u != 0u || g.n % 16u != 0u || g.k % 128u != 0u || g.k < 256u || g.k >= (1u << 30) || !dwords
           || gemmMxBlockedUsesLargeTile(g))
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        // What the re-ordering launch costs (1.5 to 3 us on operands from HBM) against what the scattered scale loads and the
        // stores of the packed order cost in the main loop.  On the ring of four that grows with the rows a tile has and with K:
        // 48 x 14336 x 4096 26.1 -> 23.1 us and x 8192 x 8192 40.0 -> 37.1, 128 rows 27.9 -> 26.5 but 42.0 -> 43.5, 256 x 4096 x
        // 14336 68.6 -> 71.1.  On the ring of two: 384 x 7168 x 2048 24.4 -> 20.9, 1024 x 1200 x 1408 14.0 -> 12.1, but 128 x 1024 x
        // 8192 52 -> 57; with more tiles than units 4096 x 1200 x 1408 24.4 -> 21.1, 512 x 14336 x 4096 57 -> 75.
        const uint32_t units = computeUnits(), stages = g.k / 128u, tiles = ceilDiv(g.m, 128u) * ceilDiv(g.n, 128u);
        const bool     raw   = mxTakesLineTiles(g) ? stages <= (g.m <= 96u ? 64u : 44u)
                               : tiles <= units ? stages <= 30u
                                                : static_cast<uint64_t>(stages) * ceilDiv(tiles, 2u * units) <= 12u;
        if(!raw)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        TileExtras ex{};
        ex.mx = MxPacked{s.a, s.b, (g.k / 128u + 1u) / 2u, s.lda, s.ldb, packedA, packedB};
        if(dtypeIn == ROCWMMA_AMD_E4M3)
            return launchMxMid<float8_t, true>(g, ex, stream);
        if(dtypeIn == ROCWMMA_AMD_E5M2)
            return launchMxMid<bfloat8_t, true>(g, ex, stream);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

    int launchGemmBlocked(int dtypeIn, int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream,
                          TileUse use)
    {
        if(g.layoutC != ROCWMMA_AMD_ROW_MAJOR)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE; // caller transposes the problem first
        switch(dtypeIn)
        {
        case ROCWMMA_AMD_F16:
            return launchGemmBlockedF16(dtypeOut, layoutA, layoutB, g, stream, use);
        case ROCWMMA_AMD_BF16:
            return launchGemmBlockedBf16(dtypeOut, layoutA, layoutB, g, stream, use);
        case ROCWMMA_AMD_I8:
            return launchGemmBlockedI8(dtypeOut, layoutA, layoutB, g, stream, use);
        case ROCWMMA_AMD_E4M3:
        case ROCWMMA_AMD_E5M2:
            return launchGemmBlockedFp8(dtypeIn, dtypeOut, layoutA, layoutB, g, stream, use);
        case ROCWMMA_AMD_F32:
            return use == TileUse::Large ? ROCWMMA_AMD_UNSUPPORTED_TYPE : launchGemmBlockedF32(dtypeOut, layoutA, layoutB, g, stream);
        default:
            return ROCWMMA_AMD_UNSUPPORTED_TYPE;
        }
    }

    int launchGemmBlockedFused(int dtypeIn, int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream)
    {
        if(g.layoutC != ROCWMMA_AMD_ROW_MAJOR)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE; // (the bias runs along the columns of a row-major D)
        switch(dtypeIn)
        {
        case ROCWMMA_AMD_F16:
            return launchGemmFusedF16(dtypeOut, layoutA, layoutB, g, stream);
        case ROCWMMA_AMD_BF16:
            return launchGemmFusedBf16(dtypeOut, layoutA, layoutB, g, stream);
        case ROCWMMA_AMD_E4M3:
        case ROCWMMA_AMD_E5M2:
            return launchGemmFusedFp8(dtypeIn, dtypeOut, layoutA, layoutB, g, stream);
        default:
            return ROCWMMA_AMD_UNSUPPORTED_TYPE;
        }
    }

} // namespace rocwmma_amd
