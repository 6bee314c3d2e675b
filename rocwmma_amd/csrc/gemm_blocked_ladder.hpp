// Blocked GEMM for gfx950: the kernels of the rungs (gemm_blocked_rungs.hpp says which one a problem runs on).  Included
// by the translation units that instantiate them for their element types (gemm_blocked_*.hip, gemm_fused*.hip).
#ifndef ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP
#define ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP

#include "gemm_blocked_launch.hpp"
#include "gemm_blocked_rungs.hpp"

namespace rocwmma_amd
{
    namespace
    {
        template <typename Cfg>
        uint32_t tilesOf(GemmArgs const& g)
        {
            return ceilDiv(g.m, Cfg::MacroM) * ceilDiv(g.n, Cfg::MacroN);
        }

        // Configurations of the rungs for 16- and 8-bit operands.  Edges: partly filled tiles and any K.  (The same tile without
        // costs 3-10 % less: no bounds on the copies and on D; 256 x 4096 x 4096 e4m3, both row-major, NarrowLines 18.0 -> 16.0 us.
        // So every rung has both, the fused epilogue's apart.)
        //
        // 16-bit and int8 operands use 16-wide blocks (16x16x32 / 16x16x64 instructions: half the accumulator
        // traffic per flop of the 32-wide forms, 5-7 % under the power cap at 256 x 256, and 6 % faster in 128 x 128
        // tiles: 512 x 14336 x 4096 f16 77 -> 74 us).  fp8 with both operands K-contiguous uses 16x16x128 with its
        // fragments streamed column by column in the tiles with rings of two, else 32x32x64.  The rings of 64-byte stages keep
        // 32-wide blocks, one or two steps of which are such a stage.
        template <typename InT, typename OutT, typename CompT, bool AK, bool BK, bool Fused>
        struct Rungs
        {
            static constexpr bool     Fp8    = sizeof(InT) == 1u && !std::is_same<InT, int8_t>::value;
            static constexpr bool     Edge16 = !Fp8 || (AK && BK); // 16-wide blocks in the rings of two
            // blocks of 16 (or half as many of 32 where the 16-wide instruction does not fit the ring)
            static constexpr uint32_t E2 = Edge16 ? 16u : 32u, D2 = Edge16 ? 1u : 2u;
            static constexpr uint32_t E3 = Fp8 ? 32u : 16u, D3 = Fp8 ? 2u : 1u;
            static constexpr uint32_t NarrowM = BK || !AK ? 4u : 2u, NarrowN = BK || !AK ? 2u : 4u; // (of 16)
            // The third B stage of Big: copies in flight at the barrier, for operands that are both K-contiguous (whole tiles, 37 to 42
            // shapes of 64 tiles and more per type pair: 2-5 % faster, up to 17 % where one round waits for memory) and for edge
            // tiles with a K-contiguous B or a dim-major A (0-1 %, up to 11 %).  Whole tiles with a dim-major operand are 0-1.5 %
            // faster on two, edge tiles of row-major operands 0.6-2.6 %.
            static constexpr bool ExtraB(bool edges)
            {
                return edges ? (BK || !AK) : (AK && BK);
            }
            // Big on whole tiles: four waves of 128 x 128, one per SIMD, where the time of a tile is matrix work (8192^3 and 4096^3 in the
            // pairs A row / B col, A row / B row, A col / B col, A col / B row, eight waves of 64 x 128 and these: f16 834 -> 797, bf16 835 ->
            // 786, f16 870 -> 842, f16 880 -> 885 us; int8 425 -> 406, 443 -> 424, 437 -> 421, 484 -> 431).  16-bit operands that are both
            // dim-major keep the eight waves (24 LDS reads of a step are transposing ones and hold up the only wave of a SIMD), and so do
            // edge tiles (3984 x 4000 x 4080: -5 to +3 %; int8 spills) and fp8, whose fragments leave no room for a second set.
            static constexpr bool WideWaves(bool edges)
            {
                return !edges && !Fp8 && (AK || BK || sizeof(InT) == 1u);
            }
            // Wide (256 x 128) likewise on four waves of 128 x 64, with the ring one stage deeper (all of the LDS): three quarters of the LDS
            // reads, copies spread over the stage.  Where A is K-contiguous, partly filled tiles too; eight waves of 64 x 64 and these:
            // 512 x 14336 x 4096 f16 with GELU 69.0 -> 65.1 us, 768 x 5504 x 4096 f16 46.6 -> 44.8, A row / B row 51.9 -> 48.5, 2000 x 3056 x
            // 1360 bf16 23.8 -> 23.1, 24.4 -> 22.6, int8 768 x 5504 x 8192 46.8 -> 44.7, 53.2 -> 48.9.  With a dim-major A it loses
            // as much as it gains (0.96 to 1.05, with C read in 16 bits 1.27): transposing reads hold up the only wave of a SIMD.
            static constexpr bool WideHalves = AK && !Fp8;
            template <uint32_t WavesM, uint32_t WavesN, uint32_t M, uint32_t N, uint32_t Stages, uint32_t PerSimd, uint32_t Edge, bool Edges, uint32_t StageKB = 0u,
                      bool Extra = false>
            using Config = BlockedConfig<InT, OutT, CompT, AK, BK, WavesM, WavesN, M, N, Stages, PerSimd, Edge, Edges, false, Fused, StageKB, Extra>;

            template <Rung R, bool Edges>
            static constexpr auto select()
            {
                if constexpr(R == Rung::Big && WideWaves(Edges))
                    return Config<2, 2, 8, 8, 2, 1, 16, false, 0, true>{};
                else if constexpr(R == Rung::Big)
                    return Config<4, 2, 4 / D2, 8 / D2, 2, 2, E2, Edges, 0, ExtraB(Edges)>{};
                else if constexpr(R == Rung::Wide && WideHalves)
                    return Config<2, 2, 8, 4, 3, 1, 16, Edges, 0, true>{};
                else if constexpr(R == Rung::Wide)
                    return Config<4, 2, 4 / D3, 4 / D3, 3, 2, E3, Edges>{};
                else if constexpr(R == Rung::Mid)
                    return Config<2, 2, 4 / D2, 4 / D2, 2, 2, E2, Edges, 0, true>{};
                else if constexpr(R == Rung::MidLines)
                    return Config<2, 2, 4 / D3, 4 / D3, 4, 1, E3, Edges, 128>{};
                else if constexpr(R == Rung::Ring2)
                    return Config<2, 2, 2, 2, 2, 2, 32, Edges>{};
                else if constexpr(R == Rung::Ring4)
                    return Config<2, 2, 2, 2, 4, 2, 32, Edges>{};
                else if constexpr(R == Rung::NarrowLines)
                    return Config<2, 2, NarrowM / D3, NarrowN / D3, 4, 1, E3, Edges, 128>{};
                else if constexpr(R == Rung::Narrow)
                    return Config<2, 2, NarrowM / D3, NarrowN / D3, 3, 2, E3, Edges>{};
                else if constexpr(R == Rung::Narrow64)
                    return Config<2, 2, NarrowM / 2, NarrowN / 2, 4, 3, 32, Edges>{};
                else if constexpr(R == Rung::Tiny)
                    return Config<2, 2, 2 / D3, 2 / D3, 4, 2, E3, Edges, 128>{};
                else
                    return Config<2, 2, 1, 1, 4, 4, 32, Edges>{};
            }
            template <Rung R, bool Edges>
            using Of = decltype(select<R, Edges>());
            // Big's rows and pipeline with half the columns, for the tiles of a last round that would be at most half full
            using HalfOfBig = std::conditional_t<WideWaves(false), Config<2, 2, 8, 4, 2, 1, 16, false, 0, true>,
                                                 Config<4, 2, 4 / D2, 4 / D2, 2, 2, E2, false, 0, ExtraB(false)>>;
        };

        template <typename InT>
        constexpr OperandKind operandKind()
        {
            return sizeof(InT) == 2u ? OperandKind::Half : (std::is_same<InT, int8_t>::value ? OperandKind::Int8 : OperandKind::Fp8);
        }

        // One problem with a row-major C/D and 16- or 8-bit operands.  AK / BK: K is the contiguous index of A (row-major) /
        // of B (col-major).  Fused: bias and activation in the epilogue (ex.fused).  ROCWMMA_AMD_UNSUPPORTED_SHAPE where one block
        // per wave is the faster way (use == TileUse::Any only).
        template <typename InT, typename OutT, typename CompT, bool AK, bool BK, bool Fused>
        int pickTile(GemmArgs const& g, hipStream_t stream, TileUse use, TileExtras const& ex)
        {
            using R                     = Rungs<InT, OutT, CompT, AK, BK, Fused>;
            constexpr uint32_t    pair  = layoutPair(AK, BK);
            constexpr OperandKind kind  = operandKind<InT>();
            using Aligned               = typename R::template Of<Rung::Big, false>;
            if(use == TileUse::Large)
                return launchCfg<Aligned>(g, stream, ex);
            const uint64_t kBytes = static_cast<uint64_t>(g.k) * sizeof(InT);
            const Rung     best   = use == TileUse::Any && g.rung != 0u
                                        ? static_cast<Rung>(g.rung)
                                        : cheapestRung(kind, pair, g.m, g.n, kBytes, sizeof(OutT), computeUnits(), use == TileUse::Any && waveTileTakes(g));
            if(best == Rung::WaveTile)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            // A rung refuses a problem whose operand rows span more than a copy's window (ROCWMMA_AMD_UNSUPPORTED_SHAPE): the smaller
            // tiles and stages behind it then have their turn.
            int  rc  = ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            bool due = false; // the chosen rung has been reached
            auto attempt = [&](auto rungC) {
                constexpr Rung rung = decltype(rungC)::value;
                // (the smallest windows are always there to fall back on: 64 rows of two K-contiguous operands, 64-byte stages else)
                constexpr bool last = rung == (AK && BK ? Rung::Tiny : (AK || BK ? Rung::Narrow64 : Rung::Ring4));
                if constexpr(hasRung(kind, pair, rung) || last)
                {
                    due = due || rung == best;
                    if(!due || rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                        return;
                    if constexpr(rung == Rung::Big)
                    {
                        rc = launchSplitTail<Aligned, typename R::HalfOfBig>(g, stream, ex);
                        if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                            return;
                    }
                    if constexpr(!Fused || rung == Rung::Big || rung == Rung::Wide)
                    {
                        // (256 x 128 tiles of fp8 with the fused epilogue and C: whole ones are slower in the kernel for whole tiles.  1024 x 7040 x 768
                        // e4m3, both row-major, GELU: with C 21.5 us as partly filled, 24.2 as whole tiles, without 18.0, 16.9.)
                        if(!(Fused && R::Fp8 && rung == Rung::Wide && g.beta != 0.0f))
                            rc = launchCfg<typename R::template Of<rung, false>>(g, stream, ex);
                        if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE) // (no whole tiles)
                            return;
                    }
                    rc = launchCfg<typename R::template Of<rung, true>>(g, stream, ex);
                }
            };
            attempt(std::integral_constant<Rung, Rung::Big>{});
            attempt(std::integral_constant<Rung, Rung::Wide>{});
            attempt(std::integral_constant<Rung, Rung::Mid>{});
            attempt(std::integral_constant<Rung, Rung::MidLines>{});
            attempt(std::integral_constant<Rung, Rung::Ring2>{});
            attempt(std::integral_constant<Rung, Rung::NarrowLines>{});
            attempt(std::integral_constant<Rung, Rung::Narrow>{});
            attempt(std::integral_constant<Rung, Rung::Tiny>{});
            attempt(std::integral_constant<Rung, Rung::Tiny64>{});
            attempt(std::integral_constant<Rung, Rung::Ring4>{});
            attempt(std::integral_constant<Rung, Rung::Narrow64>{});
            return rc;
        }

        // float32 operands (v_mfma_f32_32x32x2_f32, 64 clocks an instruction): bound by the matrix cores as soon as every
        // SIMD has a wave, so the tile is the one that spreads the work best.  A 128 x 128 tile takes 62 ns per K index
        // on a compute unit, a 64 x 64 one 18.4 (four of them 19 % more), whatever the layouts.  2048^3: 131 us
        // (131 TFLOP/s; one block per wave straight from global memory, which ran these before, 900 us), 1024^3
        // 24.6 us.  More waves (eight of 32 x 64 each) or deeper rings changed nothing.
        template <bool AK, bool BK>
        int pickTileF32(GemmArgs const& g, hipStream_t stream)
        {
            using Mid  = BlockedConfig<float32_t, float32_t, float32_t, AK, BK, 2, 2, 2, 2, 2, 2, 32, true>;
            using Tiny = BlockedConfig<float32_t, float32_t, float32_t, AK, BK, 2, 2, 1, 1, 2, 4, 32, true>;
            // The shortest K in 16-wide blocks (m or n no multiple of 32): one block per wave, 2.0 us + 0.0265 per K index + 0.077 per
            // thousand waves and K index, against 3.2 + 0.008 (16 x 256: K = 8 2.5 / 3.4 us, 16 2.7 / 3.3, 64 3.9 / 3.8; 80 x 1872: 8 2.6 / 3.6,
            // 32 4.1 / 3.6; 528 x 1040: 16 5.0 / 3.8)
            const float kilowaves = static_cast<float>(g.m) / 16.0f * (static_cast<float>(g.n) / 16.0f) * 1e-3f;
            if(waveTileTakes(g) && (g.m % 32u != 0u || g.n % 32u != 0u) && static_cast<float>(g.k) * (0.0185f + 0.077f * kilowaves) < 1.2f)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            const uint32_t units = computeUnits();
            const float    mid   = 62.0f * static_cast<float>(ceilDiv(tilesOf<Mid>(g), units));
            const float    tiny  = 18.4f * static_cast<float>(ceilDiv(tilesOf<Tiny>(g), units));
            if(mid < tiny)
            {
                const int rc = launchCfg<Mid>(g, stream);
                if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                    return rc;
            }
            return launchCfg<Tiny>(g, stream);
        }

        template <typename InT, typename OutT, typename CompT, bool Fused>
        int pickLayout(int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream, TileUse use)
        {
            TileExtras ex{};
            ex.fused      = FusedEpilogue{g.bias, g.activation};
            const bool ak = layoutA == ROCWMMA_AMD_ROW_MAJOR;
            const bool bk = layoutB == ROCWMMA_AMD_COL_MAJOR;
            if(ak && bk)
                return pickTile<InT, OutT, CompT, true, true, Fused>(g, stream, use, ex);
            if(ak && !bk)
                return pickTile<InT, OutT, CompT, true, false, Fused>(g, stream, use, ex);
            if(!ak && bk)
                return pickTile<InT, OutT, CompT, false, true, Fused>(g, stream, use, ex);
            return pickTile<InT, OutT, CompT, false, false, Fused>(g, stream, use, ex);
        }
    } // namespace
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP
