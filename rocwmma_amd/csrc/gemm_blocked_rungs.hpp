// Blocked GEMM for gfx950: which rung (macro tile and pipeline) a problem runs on.  Plain C++, so that the choice can be
// looked at on the host; the kernels of the rungs are made in gemm_blocked_ladder.hpp.
#ifndef ROCWMMA_AMD_CSRC_GEMM_BLOCKED_RUNGS_HPP
#define ROCWMMA_AMD_CSRC_GEMM_BLOCKED_RUNGS_HPP

#include <cstdint>

namespace rocwmma_amd
{
    // The rungs, largest tile first.  What differs is how many bytes a flop costs, how many stages of K are in flight while a
    // tile waits for memory, and how long a tile takes to start:
    //   Big         256 x 256, 8 waves (whole tiles of most pairs: 4), A ring of two stages, B ring of two or three
    //   Wide        256 x 128, ring of three, 4 waves (A K-contiguous, 16-bit and int8) or 8
    //   Mid         128 x 128, 4 waves, two workgroups per unit, A ring of two, B ring of three
    //   MidLines    128 x 128, 4 waves, one workgroup per unit, ring of four
    //   Ring2       128 x 128, 4 waves, two workgroups per unit, ring of two, 32-wide blocks
    //   Ring4       128 x 128, 4 waves, two workgroups per unit, ring of four 64-byte stages, 32-wide blocks
    //   NarrowLines 128 x 64 (64 x 128 where only A is K-contiguous), one workgroup per unit, ring of four
    //   Narrow      the same tile, two workgroups per unit, ring of three
    //   Narrow64    the same tile, three workgroups per unit, ring of four 64-byte stages, 32-wide blocks
    //   Tiny        64 x 64, two workgroups per unit, ring of four; both operands K-contiguous, as for Tiny64
    //   Tiny64      the same tile, four workgroups per unit, ring of four 64-byte stages, 32-wide blocks
    //   WaveTile    one block per wave straight from global memory (gemm_wave_tile.hip): the shortest K
    // Stages are 128 bytes of K (whole lines of a K-contiguous operand) where nothing else is said.
    enum class Rung : uint8_t
    {
        None,
        Big,
        Wide,
        Mid,
        MidLines,
        Ring2,
        Ring4,
        NarrowLines,
        Narrow,
        Narrow64,
        Tiny,
        Tiny64,
        WaveTile
    };

    enum class OperandKind : uint8_t
    {
        Half, // float16, bfloat16
        Int8,
        Fp8
    };

    // Layout pair: 0 both operands K-contiguous (A row-major, B col-major), 1 A only, 2 B only, 3 neither.
    constexpr uint32_t layoutPair(bool ak, bool bk)
    {
        return ak ? (bk ? 0u : 1u) : (bk ? 2u : 3u);
    }

    // Microseconds a rung takes: with at most one tile per compute unit
    //     start + alone * kKB + write * outBytes                   (one tile at a time: its copies' latency shows)
    // and with L tiles for the busiest unit
    //     start + L * (shared * kKB + writeShared * outBytes),
    // kKB = thousands of bytes of K per row, outBytes = bytes per element of D; `edges` times the terms of K where tiles or stages
    // are partly filled (bounds on every copy, rows that begin off a line).
    struct RungCost
    {
        Rung  rung;
        float start, alone, write, shared, writeShared, edges;
    };
    // One block per wave, blocks of 16 (m or n no multiple of 32) or 32:
    //     start + steps * kKB + waves * (fetch * kKB + store * outBytes),     waves in thousands.
    struct WaveCost
    {
        float start, steps, fetch, store;
    };

    constexpr uint32_t kMaxRungs = 8;
    struct RungTable
    {
        RungCost rungs[kMaxRungs]; // (Rung::None behind the last)
        WaveCost wave16, wave32;
    };

#include "gemm_blocked_costs.inc"

    constexpr bool hasRung(OperandKind kind, uint32_t pair, Rung rung)
    {
        for(uint32_t i = 0; i < kMaxRungs; ++i)
            if(kRungTables[static_cast<uint32_t>(kind)][pair].rungs[i].rung == rung)
                return true;
        return false;
    }

    constexpr uint32_t tileRows(Rung rung, uint32_t pair)
    {
        switch(rung)
        {
        case Rung::Big:
        case Rung::Wide:
            return 256u;
        case Rung::NarrowLines:
        case Rung::Narrow:
        case Rung::Narrow64:
            return pair == 1u ? 64u : 128u;
        case Rung::Tiny:
        case Rung::Tiny64:
            return 64u;
        default:
            return 128u;
        }
    }
    constexpr uint32_t tileCols(Rung rung, uint32_t pair)
    {
        switch(rung)
        {
        case Rung::Big:
            return 256u;
        case Rung::NarrowLines:
        case Rung::Narrow:
        case Rung::Narrow64:
            return pair == 1u ? 128u : 64u;
        case Rung::Tiny:
        case Rung::Tiny64:
            return 64u;
        default:
            return 128u;
        }
    }

    // Whether the problem is whole tiles and stages, and long enough for the ring.
    constexpr bool fillsTiles(Rung rung, uint32_t pair, uint32_t m, uint32_t n, uint64_t kBytes)
    {
        const bool     half  = rung == Rung::Ring4 || rung == Rung::Narrow64 || rung == Rung::Tiny64;
        const uint32_t stage = half ? 64u : 128u;
        const uint32_t ahead = half || rung == Rung::MidLines || rung == Rung::NarrowLines || rung == Rung::Tiny ? 3u
                               : rung == Rung::Wide || rung == Rung::Narrow                                      ? 2u
                                                                                                                 : 1u;
        return m % tileRows(rung, pair) == 0u && n % tileCols(rung, pair) == 0u && kBytes % stage == 0u && kBytes >= ahead * stage;
    }

    constexpr float rungTime(RungCost const& c, uint32_t pair, uint32_t m, uint32_t n, float kKB, float outBytes, uint32_t units, bool edges)
    {
        if(edges)
            kKB *= c.edges;
        const uint32_t rows = tileRows(c.rung, pair), cols = tileCols(c.rung, pair);
        const uint64_t tiles = (static_cast<uint64_t>(m) + rows - 1u) / rows * ((static_cast<uint64_t>(n) + cols - 1u) / cols);
        if(tiles <= units)
            return c.start + c.alone * kKB + c.write * outBytes;
        float load = static_cast<float>((tiles + units - 1u) / units);
        // (whole 256 x 256 tiles: a last round that would be at most half full runs as half tiles)
        const uint64_t rest = tiles % units;
        if(c.rung == Rung::Big && m % 256u == 0u && n % 256u == 0u && rest != 0u && 2u * rest <= units)
            load -= 0.4f;
        return c.start + load * (c.shared * kKB + c.writeShared * outBytes);
    }
    constexpr float waveTileTime(RungTable const& t, uint32_t m, uint32_t n, float kKB, float outBytes)
    {
        const bool      wide = m % 32u == 0u && n % 32u == 0u;
        WaveCost const& c    = wide ? t.wave32 : t.wave16;
        const float     edge = wide ? 32.0f : 16.0f, waves = static_cast<float>(m) / edge * (static_cast<float>(n) / edge) * 1e-3f;
        return c.start + c.steps * kKB + waves * (c.fetch * kKB + c.store * outBytes);
    }

    // The rung with the least estimated time (which goes to *estimate).  waveTile: one block per wave may be chosen.
    constexpr Rung cheapestRung(OperandKind kind, uint32_t pair, uint32_t m, uint32_t n, uint64_t kBytes, uint32_t outBytes, uint32_t units,
                                bool waveTile, float* estimate = nullptr)
    {
        RungTable const& table = kRungTables[static_cast<uint32_t>(kind)][pair];
        const float      kKB = static_cast<float>(kBytes) * 1e-3f, out = static_cast<float>(outBytes);
        Rung             best = Rung::None;
        float            time = 0.0f;
        for(uint32_t i = 0; i < kMaxRungs && table.rungs[i].rung != Rung::None; ++i)
        {
            const Rung  rung = table.rungs[i].rung;
            const float t    = rungTime(table.rungs[i], pair, m, n, kKB, out, units, !fillsTiles(rung, pair, m, n, kBytes));
            if(best == Rung::None || t < time)
            {
                best = rung;
                time = t;
            }
        }
        const float wave = waveTile && kBytes <= kWaveTileMaxBytes ? waveTileTime(table, m, n, kKB, out) : time;
        if(wave < time)
        {
            best = Rung::WaveTile;
            time = wave;
        }
        if(estimate)
            *estimate = time;
        return best;
    }
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_BLOCKED_RUNGS_HPP
