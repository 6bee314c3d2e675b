// Blocked GEMM for gfx950: which macro tile a problem runs on.  Included by the translation units that instantiate
// the rungs for their element types (gemm_blocked_*.hip, gemm_fused*.hip).
#ifndef ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP
#define ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP

#include "gemm_blocked_launch.hpp"

namespace rocwmma_amd
{
    namespace
    {
        // What a rung costs, fitted to timings of every rung at 60 shapes per element type and layout pair (m, n, k from
        // 16 to 14336 in steps of 16, operands from HBM).  A compute unit that runs L tiles takes
        //     L = 1:  start + alone * kKB            (one tile at a time: its copies' latency shows)
        //     L > 1:  start + L * (perTile * outBytes + shared * kKB)
        // microseconds, kKB = thousands of bytes of K per row, outBytes = bytes per element of D (results are written
        // behind the main loop).  Picked by the least of these the ladder is within 1-2 % of the best rung on average
        // (worst 18 %); occupancy thresholds alone, which this replaced, were up to 40 % off between them.
        struct RungCost
        {
            float start, alone, shared, perTile;
        };
        inline float rungTime(RungCost const& c, uint32_t tiles, uint32_t units, float kKB, float outBytes)
        {
            const float load = static_cast<float>((tiles + units - 1u) / units);
            return c.start + (tiles <= units ? c.alone * kKB : load * (c.perTile * outBytes + c.shared * kKB));
        }
        template <typename Cfg>
        uint32_t tilesOf(GemmArgs const& g)
        {
            return ceilDiv(g.m, Cfg::MacroM) * ceilDiv(g.n, Cfg::MacroN);
        }

        // One problem with a row-major C/D and 16- or 8-bit operands.  AK / BK: K is the contiguous index of A (row-major) /
        // of B (col-major).  Fused: bias and activation in the epilogue (ex.fused).
        //
        // The rungs, largest tile first.  All copy whole 128-byte lines of K per row; what differs is how many bytes
        // a flop costs (a compute unit takes at most 64 bytes a clock from its L2, so 128 x 128 tiles are bound by their
        // copies, 256 x 256 tiles are not) and how many stages are in flight while a tile waits for memory:
        //   Big    256 x 256, 8 waves, A ring of two stages, B ring of three (all 160 KiB of LDS).  The third B stage keeps
        //          copies in flight at the barrier: 512 x 14336 x 4096 f16 99 -> 90 us, int8 4096 x 14336 x 4096 1.5 %.  Whole tiles with
        //          a dim-major operand keep two (8192^3 bf16 0.5-0.7 % faster in both such pairs with one).
        //   Wide   256 x 128, 8 waves, ring of three (144 KiB): 512 x 14336 x 4096 f16 77 -> 63 us against 128 x 128 tiles on
        //          the ring of two, int8 43 -> 34; on a ring of two of its own it was 82.
        //   Mid    128 x 128, 4 waves, two workgroups per unit with 80 KiB each (A ring of two, B ring of three):
        //          2048^3 f16 25.5 -> 22.4 us, 512 x 14336 x 4096 77 -> 69 against rings of two.
        //   Narrow 128 x 64 (64 x 128 where only A is K-contiguous), ring of three, two workgroups per unit;
        //          fp8 also on a ring of four with one workgroup per unit (three stages of 24 KiB in flight).
        //   Tiny   64 x 64, ring of four, two workgroups per unit; both operands K-contiguous (a dim-major LDS tile is
        //          at least 128 wide).
        // 16-bit and int8 operands use 16-wide blocks (16x16x32 / 16x16x64 instructions: half the accumulator
        // traffic per flop of the 32-wide forms, 5-7 % under the power cap at 256 x 256, and 6 % faster in 128 x 128
        // tiles: 512 x 14336 x 4096 f16 77 -> 74 us).  fp8 with both operands K-contiguous uses 16x16x128 with its
        // fragments streamed column by column in the tiles with rings of two, else 32x32x64.
        // Every rung but Aligned takes partly filled tiles at the edges and any K (Edges).
        template <typename InT, typename OutT, typename CompT, bool AK, bool BK, bool Fused>
        int pickTile(GemmArgs const& g, hipStream_t stream, bool forceLargeTile, TileExtras const& ex)
        {
            static constexpr bool Fp8    = sizeof(InT) == 1u && !std::is_same<InT, int8_t>::value;
            static constexpr bool Edge16 = !Fp8 || (AK && BK); // 16-wide blocks in the rings of two
            // blocks of 16 (or half as many of 32 where the 16-wide instruction does not fit the ring)
            static constexpr uint32_t E2 = Edge16 ? 16u : 32u, D2 = Edge16 ? 1u : 2u;
            static constexpr uint32_t E3 = Fp8 ? 32u : 16u, D3 = Fp8 ? 2u : 1u;
            using Aligned = BlockedConfig<InT, OutT, CompT, AK, BK, 4, 2, 4 / D2, 8 / D2, 2, 2, E2, false, false, Fused, 0, AK && BK>;
            // same rows and pipeline with half the columns, for the tiles of a last round that would be at most half full
            using AlignedHalf = BlockedConfig<InT, OutT, CompT, AK, BK, 4, 2, 4 / D2, 4 / D2, 2, 2, E2, false, false, Fused, 0, AK && BK>;
            using Big    = BlockedConfig<InT, OutT, CompT, AK, BK, 4, 2, 4 / D2, 8 / D2, 2, 2, E2, true, false, Fused, 0, true>;
            using Wide   = BlockedConfig<InT, OutT, CompT, AK, BK, 4, 2, 4 / D3, 4 / D3, 3, 2, E3, true, false, Fused>;
            using Mid    = BlockedConfig<InT, OutT, CompT, AK, BK, 2, 2, 4 / D2, 4 / D2, 2, 2, E2, true, false, Fused, 0, true>;
            static constexpr uint32_t NarrowM = BK ? 4u : 2u, NarrowN = BK ? 2u : 4u;
            using Narrow = BlockedConfig<InT, OutT, CompT, AK, BK, 2, 2, NarrowM / D3, NarrowN / D3, 3, 2, E3, true, false, Fused>;
            using NarrowLines = BlockedConfig<InT, OutT, CompT, AK, BK, 2, 2, NarrowM / D3, NarrowN / D3, 4, 1, E3, true, false, Fused, 128>;
            using Tiny   = BlockedConfig<InT, OutT, CompT, AK, BK, 2, 2, 2 / D3, 2 / D3, 4, 2, E3, true, false, Fused, 128>;

            const bool aligned = g.m % Aligned::MacroM == 0u && g.n % Aligned::MacroN == 0u && g.k % Aligned::MacroK == 0u
                                 && g.k >= Aligned::MacroK;
            if(forceLargeTile)
                return aligned ? launchCfg<Aligned>(g, stream, ex) : ROCWMMA_AMD_UNSUPPORTED_SHAPE;

            constexpr bool     Byte      = sizeof(InT) == 1u;
            constexpr RungCost BigCost  = AK && BK   ? RungCost{7.5f, 8.1f, 11.6f, 3.0f}
                                          : AK != BK ? RungCost{7.5f, 9.6f, 12.4f, 3.2f}
                                                     : RungCost{7.0f, 9.6f, 13.4f, 2.9f};
            constexpr RungCost WideCost = AK && BK   ? RungCost{6.0f, Byte ? 4.5f : 5.1f, Byte ? 6.6f : 6.9f, Byte ? 2.2f : 1.7f}
                                          : AK != BK ? RungCost{6.3f, Byte ? 5.4f : 5.8f, 6.9f, 2.6f}
                                                     : RungCost{5.5f, 6.4f, 7.8f, 2.7f};
            constexpr RungCost MidCost  = AK && BK   ? RungCost{5.2f, Byte ? 3.2f : 3.6f, Byte ? 3.55f : 3.7f, 0.85f}
                                          : AK != BK ? RungCost{5.3f, Byte ? 3.9f : 4.5f, 3.85f, 0.87f}
                                                     : RungCost{4.6f, 4.85f, 4.12f, 0.95f};
            constexpr RungCost NarrowCost = AK && BK ? RungCost{5.2f, Byte ? 2.05f : 2.5f, Byte ? 2.3f : 2.5f, 0.42f}
                                                     : RungCost{4.9f, Byte ? 3.0f : 3.35f, Byte ? 3.7f : 2.95f, 0.4f};
            constexpr RungCost LinesCost = AK && BK ? RungCost{5.5f, 1.77f, 2.56f, 0.52f} : RungCost{5.1f, 2.75f, 4.05f, 0.48f};
            constexpr RungCost TinyCost  = RungCost{5.1f, Byte ? 1.45f : 1.95f, Byte ? 1.6f : 1.75f, 0.14f};

            const uint32_t units = computeUnits(); // (once: it asks the runtime for the current device)
            const float    kKB = static_cast<float>(g.k) * (sizeof(InT) * 1e-3f), outBytes = sizeof(OutT);
            enum Rung
            {
                kBig,
                kWide,
                kMid,
                kNarrow,
                kLines,
                kTiny
            };
            Rung  best = kBig;
            float time = rungTime(BigCost, tilesOf<Big>(g), units, kKB, outBytes);
            if(aligned)
            {
                // a last round that would be at most half full runs as half tiles (launchSplitTail)
                const uint32_t tiles = tilesOf<Big>(g), rest = tiles % units;
                if(tiles > units && rest != 0u && 2u * rest <= units)
                    time -= 0.4f * (BigCost.perTile * outBytes + BigCost.shared * kKB);
            }
            auto consider = [&](Rung r, RungCost const& c, uint32_t tiles) {
                const float t = rungTime(c, tiles, units, kKB, outBytes);
                if(t < time)
                {
                    time = t;
                    best = r;
                }
            };
            consider(kWide, WideCost, tilesOf<Wide>(g));
            consider(kMid, MidCost, tilesOf<Mid>(g));
            if constexpr(AK || BK)
                consider(kNarrow, NarrowCost, tilesOf<Narrow>(g));
            if constexpr(Fp8 && (AK || BK))
                consider(kLines, LinesCost, tilesOf<NarrowLines>(g));
            if constexpr(AK && BK)
                consider(kTiny, TinyCost, tilesOf<Tiny>(g));
            if(best == kBig)
            {
                int rc = ROCWMMA_AMD_UNSUPPORTED_SHAPE;
                if(aligned)
                {
                    rc = launchSplitTail<Aligned, AlignedHalf>(g, stream, ex);
                    if(rc == ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                        rc = launchCfg<Aligned>(g, stream, ex);
                }
                else
                    rc = launchCfg<Big>(g, stream, ex);
                if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE) // (an operand's tile rows span more than a copy's window)
                    return rc;
            }
            if(best == kWide)
            {
                const int rc = launchCfg<Wide>(g, stream, ex);
                if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE)
                    return rc;
            }
            if constexpr(AK || BK)
            {
                if(best == kNarrow)
                    return launchCfg<Narrow>(g, stream, ex);
            }
            if constexpr(Fp8 && (AK || BK))
            {
                if(best == kLines)
                    return launchCfg<NarrowLines>(g, stream, ex);
            }
            if constexpr(AK && BK)
            {
                if(best == kTiny)
                    return launchCfg<Tiny>(g, stream, ex);
            }
            return launchCfg<Mid>(g, stream, ex);
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
        int pickLayout(int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream, bool forceLargeTile)
        {
            TileExtras ex{};
            ex.fused      = FusedEpilogue{g.bias, g.activation};
            const bool ak = layoutA == ROCWMMA_AMD_ROW_MAJOR;
            const bool bk = layoutB == ROCWMMA_AMD_COL_MAJOR;
            if(ak && bk)
                return pickTile<InT, OutT, CompT, true, true, Fused>(g, stream, forceLargeTile, ex);
            if(ak && !bk)
                return pickTile<InT, OutT, CompT, true, false, Fused>(g, stream, forceLargeTile, ex);
            if(!ak && bk)
                return pickTile<InT, OutT, CompT, false, true, Fused>(g, stream, forceLargeTile, ex);
            return pickTile<InT, OutT, CompT, false, false, Fused>(g, stream, forceLargeTile, ex);
        }
    } // namespace
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_BLOCKED_LADDER_HPP
