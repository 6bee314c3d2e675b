// Blocked GEMM for gfx950, device side: D = alpha * A * B + beta * C, C/D row-major.  Shared by the
// one-tile-per-workgroup kernel (gemm_blocked.hip) and the persistent stream-K kernel
// (gemm_streamk.hip).
//
// The workload of the reference's perf_hgemm sample (gemm_rocwmma_d,
// samples/perf_hgemm.cpp:518-714: macro tile per workgroup, wave tile of MFMA blocks per wave,
// two LDS buffers, next K slab prefetched while the current one is multiplied), re-tiled and
// re-plumbed for CDNA4:
//
//   reference (gfx9 params)                      this kernel (256 x 256 configuration)
//   macro tile 128 x 128 x 16, 4 waves           256 x 256 x (128 bytes of K) x ring of two LDS stages, 8 waves
//                                                (two per SIMD: one keeps the matrix pipe fed while the
//                                                other issues the stage's copies or waits at the barrier)
//   wave tile 2 x 2 blocks of 32x32x16 (2 MFMA)  4 x 8 blocks of 16x16, wide-K MFMAs (16x16x32 f16 / bf16,
//                                                16x16x64 int8, 16x16x128 fp8), 64 per wave and stage
//   global -> VGPR -> shuffle -> LDS             global -> LDS directly (buffer_load_dwordx4 ... lds), issued by
//                                                the first wave of each SIMD for itself and its partner
//   LDS -> VGPR -> shuffle (AOS<->SOA)           swizzled ds_read_b128, or ds_read_b64_tr_b16 / _b8
//                                                for operands whose K is not contiguous
//   2 LDS buffers, wait + barrier per step       copies one stage ahead, one barrier per 128-byte stage
//   8 MFMA between barriers                      64 MFMA (1024 clocks of matrix-pipe work) per wave between barriers
//   C read / D written in fragment layout       C staged through LDS (full-row non-temporal
//                                                copies), D written in fragment layout
//   grid (m/128, n/128)                          1-D grid, tiles dealt to XCDs in L2-friendly patches
//                                                (9 % faster than the plain order at 8192^3)
//
// The smaller configurations (256 x 128 tiles of 8 waves; 128 x 128, 128 x 64, 64 x 64 tiles of 4) come with rings of two, three
// and four such stages, the ring of B perhaps a stage deeper than that of two of A, or with a ring of four stages of 64 bytes
// (copies three stages ahead).
//
// Column-major C/D is handled by the caller as the transposed problem (D^T = B^T A^T).
#ifndef ROCWMMA_AMD_CSRC_GEMM_BLOCKED_CORE_HPP
#define ROCWMMA_AMD_CSRC_GEMM_BLOCKED_CORE_HPP

#include "common.hpp"
#include "copy_waits.hpp"
#include <rocwmma/rocwmma_lds.hpp>

using namespace rocwmma;

namespace rocwmma_amd
{
    namespace
    {
        constexpr uint32_t kXcds = 8; // MI355X: 8 accelerator complex dies, one L2 each

        template <typename InT_,
                  typename OutT_,
                  typename CompT_,
                  bool     AKMajor_, // A row-major  (K contiguous)
                  bool     BKMajor_, // B col-major  (K contiguous)
                  uint32_t WavesM_,
                  uint32_t WavesN_,
                  uint32_t BlocksM_,
                  uint32_t BlocksN_,
                  uint32_t Stages_       = 4u, // LDS ring depth
                  uint32_t WavesPerSimd_ = 1u, // waves per SIMD: sizes the register budget, and no more become resident
                  uint32_t BlockEdge_    = 32u, // MFMA block edge: 32 (32x32xK) or 16 (16x16x2K)
                  bool     Edges_        = false, // M, N and K need not fill whole macro tiles and stages (multiples of 16, 32 bytes do)
                  bool     Scaled_       = false, // fp8 operands with one E8M0 scale per 32 elements of K (MX)
                  bool     Fused_        = false, // epilogue adds a per-column bias and applies an activation
                  uint32_t StageKB_      = 0u, // bytes of K per stage (0: 64 in the ring of four, else 128)
                  bool     ExtraB_       = false, // the ring of B is one stage deeper than the ring of A
                  bool     RawScales_    = false> // Scaled, 32-wide blocks: the scales as the caller has them (see MxPacked)
        struct BlockedConfig
        {
            using InT   = InT_;
            using OutT  = OutT_;
            using CompT = CompT_;

            static constexpr bool     AKMajor = AKMajor_;
            static constexpr bool     BKMajor = BKMajor_;
            // Partly filled tiles at the lower and right edges of C/D: operand reads past a matrix end
            // are cut off by the buffer bounds (rows and columns beyond the problem only ever meet
            // results beyond it), C reads and D stores are masked lane by lane.  Along K the copies of a
            // last, partly filled stage (and of stages beyond it) read nothing past the end of K and
            // store zeros for both operands.
            static constexpr bool     Edges   = Edges_;
            // Block-scaled operands: the scaled instruction's K order decides which bytes a lane holds
            // (two runs of 16 from the two halves of the stage, see rocwmma/internal/fragment_map.hpp),
            // so the fragments are read like two steps of a 16-bytes-per-lane operand.
            static constexpr bool     Scaled  = Scaled_;
            static constexpr bool     RawScales = RawScales_;
            // (block scales come with K in whole stages: 64 x 4096 x 4096 e4m3 27.1 us with the K bounds, 26.4 without)
            static constexpr bool     EdgesK  = Edges_ && !Scaled_;
            // D = act(alpha * A * B + beta * C + bias[column]): see FusedEpilogue
            static constexpr bool     Fused   = Fused_;
            static constexpr uint32_t WavesM  = WavesM_;
            static constexpr uint32_t WavesN  = WavesN_;
            static constexpr uint32_t BlocksM = BlocksM_;
            static constexpr uint32_t BlocksN = BlocksN_;
            static constexpr uint32_t Waves   = WavesM * WavesN;
            static constexpr uint32_t Threads = Waves * 64u;
            static constexpr uint32_t Block   = BlockEdge_; // MFMA edge
            static constexpr uint32_t WaveM   = BlocksM * Block;
            static constexpr uint32_t WaveN   = BlocksN * Block;
            static constexpr uint32_t MacroM  = WavesM * WaveM;
            static constexpr uint32_t MacroN  = WavesN * WaveN;
            // bytes of K per pipeline stage: 128 (whole lines of a K-contiguous operand), 64 in the ring of four that does not say
            // otherwise
            static constexpr uint32_t StageKB = StageKB_ != 0u ? StageKB_ : (Stages_ == 4u ? 64u : 128u);
            static constexpr uint32_t MacroK  = StageKB / sizeof(InT); // K elements per stage

            // Fragments of one MFMA step.  BlockK = K of the widest single instruction.
            // (float32: the instruction takes one float per lane; a lane holds 16 bytes of K and feeds four
            // instructions from them, the same four K indices for both operands, so their order does not matter)
            static constexpr uint32_t KPack      = sizeof(InT) == 4u ? 4u : detail::maxKPack(detail::packClassOf<InT>());
            static constexpr uint32_t BlockK     = KPack * (64u / Block); // 2 (32-wide) or 4 (16-wide) lane groups along K
            static constexpr uint32_t KPackBytes = KPack * sizeof(InT);
            static constexpr uint32_t KSteps     = MacroK / BlockK; // MFMA steps per stage (1 or 2)

            using FragA   = fragment<matrix_a, Block, Block, BlockK, InT, row_major>;
            using FragB   = fragment<matrix_b, Block, Block, BlockK, InT, col_major>;
            using FragAcc = fragment<accumulator, Block, Block, BlockK, CompT>;
            using FragC   = fragment<accumulator, Block, Block, BlockK, OutT, row_major>;

            // (a dim-major tile holds one K index per LDS row: StageKB / sizeof(InT) rows)
            template <uint32_t Dim>
            using DimTile = std::conditional_t<
                sizeof(InT) == 4u, lds::DimMajorTile32<Dim, StageKB / 4u>,
                std::conditional_t<sizeof(InT) == 2u, lds::DimMajorTile<Dim % 128u == 0u ? Dim : 128u, StageKB / 2u>,
                                   lds::DimMajorTile8<(Dim == 128u || Dim == 256u) ? Dim : 128u, StageKB>>>;
            // (16-wide blocks with 32 bytes of K per lane, fp8 16x16x128: the K-major tile's pair reader)
            static constexpr bool PairReads = Block == 16u && KPackBytes == 32u && !Scaled;
            using TileA = std::conditional_t<AKMajor, lds::KMajorTile<MacroM, StageKB, PairReads>, DimTile<MacroM>>;
            using TileB = std::conditional_t<BKMajor, lds::KMajorTile<MacroN, StageKB, PairReads>, DimTile<MacroN>>;

            static constexpr uint32_t BytesA     = MacroM * StageKB;
            static constexpr uint32_t BytesB     = MacroN * StageKB;
            static constexpr uint32_t StageBytes = BytesA + BytesB;
            static constexpr uint32_t Stages     = Stages_; // ring of K stages in LDS
            static constexpr uint32_t WavesPerSimd = WavesPerSimd_;
            static constexpr uint32_t StagesB = Stages_ + (ExtraB_ ? 1u : 0u);
            // LDS: stage by stage, A in front of B (one address serves both operands); with an extra B stage the ring of A, then the
            // ring of B
            static constexpr uint32_t StrideA = ExtraB_ ? BytesA : StageBytes;
            static constexpr uint32_t StrideB = ExtraB_ ? BytesB : StageBytes;
            static constexpr uint32_t FirstB  = ExtraB_ ? Stages * BytesA : BytesA;
            static constexpr uint32_t LdsBytes   = Stages * BytesA + StagesB * BytesB;
            static constexpr uint32_t CopiesA    = BytesA / 1024u / Waves; // direct copies per wave per stage
            static constexpr uint32_t CopiesB    = BytesB / 1024u / Waves;
            static constexpr uint32_t Copies     = CopiesA + CopiesB;
            // With two waves per SIMD only the first wave of each SIMD issues the copies of the main loop, for
            // itself and for its partner (wave + CopyWaves).  A copy holds its wave's instruction issue for a
            // dozen cycles; when both waves of a SIMD issue theirs at the same point of the same phase
            // nothing feeds the matrix pipe meanwhile, with one issuer the partner's MFMAs fill that time
            // (8192^3, A row-major / B col-major: f16 0.845 -> 0.798 ms, bf16 0.821 -> 0.765; both row-major
            // 0.906 -> 0.884, both col-major 0.883 -> 0.853; with the second wave of each SIMD as the issuer
            // 1-5 % slower than that).  A col-major / B row-major (neither K-contiguous: every fragment comes
            // from transposing reads) is left as it was: 5 % slower with one issuer.  So are the kernels with
            // block scales: their main loop loads scales into registers, and behind a branch that only some
            // waves take the compiler waits for every copy in flight before it uses them (five times slower).
            // Wave tiles of 128 rows, one wave per SIMD (the loop is at Cfg::WideWave below): the accumulators take 256 registers, so they
            // live in the accumulation half of the register file.
            static constexpr bool     WideWave = WavesPerSimd_ == 1u && BlocksM_ == 8u && BlockEdge_ == 16u && ExtraB_;
            static constexpr uint32_t CopyWaves
                = (Waves == 8u && WavesPerSimd_ == 2u && (Stages_ == 2u || Stages_ == 3u) && (AKMajor || BKMajor) && !Scaled_) ? 4u : Waves;
            // LDS read instructions per MFMA step: b128 reads per block (K-major) or two transposing b64 reads
            static constexpr uint32_t TrReads      = KPackBytes / 8u; // transposing 8-byte reads (float32: reads of two dwords) per operand
            static constexpr uint32_t ReadsA       = BlocksM * (AKMajor ? KPackBytes / 16u : TrReads);
            static constexpr uint32_t ReadsB       = BlocksN * (BKMajor ? KPackBytes / 16u : TrReads);
            static constexpr uint32_t ReadsPerStep = ReadsA + ReadsB;
            static constexpr uint32_t MfmasPerStep = BlocksM * BlocksN;
            // beta * C operand staged through LDS in the epilogue, in groups of Block rows by
            // GroupBlocks blocks (256- or 512-byte rows)
            static constexpr uint32_t GroupBlocks
                = (WaveN == 128u && 2u * Block * 128u * sizeof(OutT) * Waves <= LdsBytes) ? 128u / Block : 64u / Block;
            static constexpr bool StagedC = sizeof(OutT) == 4u && WaveN % 64u == 0u
                                            && BlocksM * (BlocksN / GroupBlocks) >= 2u
                                            && 2u * Block * GroupBlocks * Block * sizeof(OutT) * Waves <= LdsBytes;

            // group buffers per wave: four for wide waves, which are half as many (with two, 4096^3 bf16 with C took as long as with eight
            // waves, 127.2 against 126.7 us; with four 122.1 against 128.1), two else
            static constexpr uint32_t BuffersC = WideWave && 4u * Block * GroupBlocks * Block * sizeof(OutT) * Waves <= LdsBytes ? 4u : 2u;

            // Partly filled 256 x 256 tiles of fp8, both operands row-major, with the fused epilogue: the compiler left the descriptors of the
            // copies in vector registers, and every copy was a loop over the lanes' descriptors (3456 x 2944 x 2816 with GELU 54.9 us, 48.5 with
            // scalar ones).
            static constexpr bool ScalarSources = Edges_ && Fused_ && BlockEdge_ == 32u && AKMajor && !BKMajor && MacroN == 256u;

            // Fused epilogue of 256 x 256 tiles on wide waves, and of their half tiles: a loop over the rows of blocks that is not unrolled (with
            // a C of 16 bits it is).  256 results per lane through bias and GELU one after the other are 37 KB of code, and what a first call, or
            // one behind other kernels, waits for is that code, with one wave per SIMD and nobody to cover it.  f16, GELU, K = 512 to 4096, operands
            // not used before, eight waves, four unrolled, four with the loop, us: 1536 x 14336 x 512 51.2, 54.9, 50.3; 2048 x 14336 x 1024 79.6, 81.3,
            // 77.4; 2048 x 7168 x 2048 70.3, 68.2, 62.1; 4096^3 117.9, 111.2, 107.7; with a C of 32 bits 2560 x 7168 x 1024 78.5, 83.9, 78.9.
            // The same operands again: 40.7, 41.9, 40.8; 72.3, 70.7, 69.8; 57.9, 55.6, 55.4; 109.7, 104.5, 103.6; 68.5, 67.2, 69.5.  128 results
            // per lane (256 x 128 tiles) gain nothing: 512 x 14336 x 4096 79.6, 80.6 unrolled, 81.4 with the loop, again 65.6, 58.3, 61.1.
            static constexpr bool RolledRows = Fused_ && WideWave && Stages_ == 2u;

            // C of the small tiles (at most 32 registers of it) is loaded in front of the main loop: behind it, the loads' latency
            // is a large part of a short problem (per call in a captured graph: 256^3 f16 4.0 -> 3.55 us, 512 x 1024 x 1024 e4m3
            // 5.4 -> 4.8, 640 x 1200 x 1360 bf16 10.0 -> 9.5).
            // (int8 results count as registers, not as bytes: the early elements are held one to a register, so the 64 x 128 wave
            // tiles of the 256 x 256 rung spilled more than a hundred registers: 3072^3 int8 -> int8 38 -> 50 us.)
            static constexpr bool PrefetchC
                = !StagedC && !Scaled && WaveM * WaveN * sizeof(OutT) <= 64u * 128u && WaveM * WaveN <= 64u * 64u;

            static_assert(Block == 32u || Block == 16u, "MFMA blocks are 32 or 16 wide");
            static_assert(!Scaled
                              || (KPackBytes == 32u && AKMajor && BKMajor && (Block == 32u || !Edges_)
                                  && (Stages_ == 2u || (Stages_ == 4u && StageKB == 128u && Block == 32u))),
                          "block scales: fp8 on K-contiguous operands in the ring of two (16x16x128 on whole tiles, or 32x32x64), "
                          "or 32x32x64 in the ring of four 128-byte stages");
            static_assert(!RawScales || (Scaled && Block == 32u && Edges), "scales in the caller's order: 32x32x64 on edge tiles");
            static_assert(Block == 32u || KPackBytes == 16u || ((PairReads || Scaled) && AKMajor && BKMajor && Stages_ == 2u),
                          "16-wide blocks: 16 bytes of K per lane (16-bit types, int8), or fp8 16x16x128 on K-contiguous "
                          "operands in the ring of two");
            static_assert(sizeof(InT) <= 4u && (sizeof(InT) != 4u || Block == 32u), "8-bit, 16-bit and (in 32-wide blocks) float32 operands");
            static_assert(sizeof(InT) != 1u || ((AKMajor || MacroM == 128u || MacroM == 256u) && (BKMajor || MacroN == 128u || MacroN == 256u)),
                          "dim-major tiles of 8-bit operands are 128 or 256 wide");
            static_assert(TileA::bytes == BytesA && TileB::bytes == BytesB, "stage geometry mismatch");
            static_assert(BytesA % (1024u * Waves) == 0u && BytesB % (1024u * Waves) == 0u,
                          "a stage must split into whole-wave copies evenly");
            static_assert((Stages - 1u) * Copies < 64u, "too many copies in flight for vmcnt");
            static_assert(Stages == 4u || StageKB == 64u || KSteps == 2u || KSteps == 4u || (KSteps == 1u && BlocksN % 2u == 0u),
                          "the ring of two runs one (fragments streamed by columns), two or four MFMA steps per stage");
            static_assert(LdsBytes <= Constants::AMDGCN_LDS_MAX_SIZE_BYTES, "macro tile does not fit the LDS");
            // the dim-major tile's swizzle looks at K row bits 0..3: a wave's copies must all start
            // on the same K row modulo 16
            // (the 8-bit tile's looks at K row bit 4 as well, the float32 tile's at bit 2 only)
            static constexpr uint32_t SwizzleRows = sizeof(InT) == 4u ? 8u : (sizeof(InT) == 2u ? 16u : 32u);
            // lane offsets that the copies of a wave take turns with, where its copies do not all start on the same K row modulo that
            static constexpr uint32_t turns(bool kMajor, uint32_t rowsPerCopy)
            {
                return kMajor || (Waves * rowsPerCopy) % SwizzleRows == 0u ? 1u : SwizzleRows / (Waves * rowsPerCopy);
            }
            static constexpr uint32_t TurnsA = turns(AKMajor, TileA::rowsPerCopy), TurnsB = turns(BKMajor, TileB::rowsPerCopy);
            static_assert(WideWave || (TurnsA == 1u && TurnsB == 1u),
                          "wave pool too small for the dim-major tile");
            // the K-major tile's swizzle looks at row bits 0..3 likewise
            static_assert((!AKMajor || (Waves * TileA::rowsPerCopy) % 16u == 0u)
                              && (!BKMajor || (Waves * TileB::rowsPerCopy) % 16u == 0u),
                          "wave pool too small for the K-major tile");
        };

        // Deals the 1-D grid to tiles so that the workgroups resident on one XCD (ids congruent
        // mod 8 land on the same XCD) form a compact patch of the tile grid and share A / B
        // panels through that XCD's L2.
        ROCWMMA_DEVICE inline void tileOfWorkgroup(uint32_t wg, uint32_t tilesM, uint32_t tilesN, uint32_t& tm, uint32_t& tn)
        {
            const uint32_t total = tilesM * tilesN;
            uint32_t       id    = wg;
            if(total % kXcds == 0u)
                id = (wg % kXcds) * (total / kXcds) + wg / kXcds;
            // panels of 4 tile rows, walked column by column: the 32 workgroups an XCD runs at a
            // time cover 4 x 8 tiles (measured: 1 % faster than 8 x 4, 5 % faster than 16 x 2)
            constexpr uint32_t panel    = 4u;
            const uint32_t     perPanel = panel * tilesN;
            const uint32_t     panelIdx = id / perPanel;
            const uint32_t     firstRow = panelIdx * panel;
            const uint32_t     rowsHere = (tilesM - firstRow) < panel ? (tilesM - firstRow) : panel;
            const uint32_t     inPanel  = id - panelIdx * perPanel;
            tm                          = firstRow + inPanel % rowsHere;
            tn                          = inPanel / rowsHere;
        }

        // Scheduling hint: within the current scheduling region, issue `Mfmas` matrix instructions
        // with `Reads` LDS reads and `Copies` global -> LDS copies spread evenly between them.
        template <uint32_t Mfmas, uint32_t Reads, uint32_t Copies>
        ROCWMMA_DEVICE ROCWMMA_INLINE void scheduleInterleaved()
        {
            constexpr uint32_t Div = Mfmas > 0u ? Mfmas : 1u; // (an empty group: the loop does not run)
#pragma unroll
            for(uint32_t j = 0; j < Mfmas; ++j)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // 1 MFMA
                const uint32_t r = ((j + 1u) * Reads) / Div - (j * Reads) / Div;
                const uint32_t c = ((j + 1u) * Copies) / Div - (j * Copies) / Div;
                if(r == 1u)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); // DS read
                else if(r == 2u)
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                else if(r > 2u)
                    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
                if(c == 1u)
                    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0); // VMEM
                else if(c >= 2u)
                    __builtin_amdgcn_sched_group_barrier(0x010, 2, 0);
            }
        }


        // Compile-time loop: f(std::integral_constant<uint32_t, 0>{}), ..., f(<N - 1>) -- for bodies whose
        // iteration index must be a constant expression (instruction immediates).
        template <typename F, uint32_t... I>
        ROCWMMA_DEVICE ROCWMMA_INLINE void staticForImpl(F&& f, std::integer_sequence<uint32_t, I...>)
        {
            (f(std::integral_constant<uint32_t, I>{}), ...);
        }
        template <uint32_t N, typename F>
        ROCWMMA_DEVICE ROCWMMA_INLINE void staticFor(F&& f)
        {
            staticForImpl(f, std::make_integer_sequence<uint32_t, N>{});
        }

        // Block scales of a Scaled configuration, in the order the lanes load them (written by the
        // re-ordering kernel in gemm_mx.hip): per operand, group of 64 rows of A (columns of B) and pair
        // of K stages, 8 bytes per lane = [block of 16 rows 0..3][stage of the pair 0..1]; lane l's bytes
        // are the scales of row l % 16 of each block and K block l / 16 of each stage.
        struct MxPacked
        {
            const void* a;
            const void* b;
            uint32_t    pairs; // pairs of stages along K (the last one padded when the stage count is odd)
            // RawScales: a and b are the caller's scales, one row of k / 32 bytes per row of A / column of B, these many
            // bytes apart (4-byte aligned).  A lane then loads the eight bytes of its row for a pair of stages as they lie.
            uint32_t    lda, ldb;
            void*       packedA; // RawScales: where the packed order is left (PairScales)
            void*       packedB;
        };

        // The packed dword of a 32-wide block and lane out of the eight scales of the lane's row for a pair of stages (lo: K blocks
        // 0..3, hi: 4..7): byte = instruction step, of which lanes 0..31 take the even K block and lanes 32..63 the odd one.
        ROCWMMA_DEVICE ROCWMMA_INLINE uint32_t packPairScales(uint32_t lo, uint32_t hi, uint32_t lane)
        {
#if ROCWMMA_ARCH_GFX950
            return __builtin_amdgcn_perm(hi, lo, lane < 32u ? 0x06040200u : 0x07050301u);
#else
            return lo ^ hi ^ lane;
#endif
        }

        // What a Fused configuration's epilogue does beyond alpha * acc + beta * C.
        struct FusedEpilogue
        {
            const float* bias; // one value per column of D (n floats), or nullptr
            int          activation; // rocwmma_amd_activation
        };

        // Per-launch arguments beyond the GEMM's own, for the configurations that use them.
        struct TileExtras
        {
            MxPacked      mx;
            FusedEpilogue fused;
        };

        // Scales of a wave's 32-wide blocks along one dimension, a pair of stages (256 bytes of K, four instruction steps) at a
        // time: one dword per block and lane, byte = step.  Raw: made from the eight bytes of the lane's row (rows past the
        // problem's get the scale 1; a last pair that is half a pair starts four bytes early), and left in the workspace in
        // the packed order all the same, as the re-ordering launch leaves them: the workspace then serves calls on packed
        // scales.  The dwords are what the lanes hold anyway, so that is a store per pair of stages: 128 x 14336 x 4096 e4m3
        // 18.6 -> 19.2 us (read again and written behind the results: 21.0; with the re-ordering launch: 20.7).  Waves that have
        // nothing to leave store past the end of an empty buffer, without a branch.
        template <typename Cfg, uint32_t Blocks>
        struct PairScales
        {
            static constexpr bool Raw = Cfg::RawScales;
            static_assert(Blocks == 1u || Blocks == 2u || (!Raw && Blocks % 2u == 0u), "a wave's blocks: one, or whole groups of two");
            uint32_t       now[Blocks] = {}, next[Raw ? 2u * Blocks : Blocks] = {};
            const char*    from[Raw ? Blocks : 1u];
            bool           inside[Raw ? Blocks : 1u]; // this lane's row of a block is one of the problem's
            uint32_t       pairs, last, lane, keepAt; // last: Raw, byte the last whole pair of a row starts at
            lds::BufferRsrc kept; // Raw: the packed scales of this wave's group of 64 rows
            ROCWMMA_DEVICE ROCWMMA_INLINE
                PairScales(const void* scales, uint32_t ld, uint32_t pairs_, uint32_t row0, uint32_t rows, uint32_t k, uint32_t lane_, void* packed, bool keeper)
                : pairs(pairs_)
                , last(k / 32u - 8u)
                , lane(lane_)
            {
                if constexpr(Raw)
                {
#pragma unroll
                    for(uint32_t b = 0; b < Blocks; ++b)
                    {
                        const uint32_t row = row0 + b * 32u + (lane & 31u);
                        inside[b]          = row < rows;
                        from[b]            = static_cast<const char*>(scales) + static_cast<size_t>(inside[b] ? row : rows - 1u) * ld;
                    }
                    char* group = static_cast<char*>(packed) + static_cast<size_t>(row0 / 64u) * pairs * 512u;
                    kept        = lds::makeSource(group, keeper && row0 / 64u * 64u < rows ? group + static_cast<size_t>(pairs) * 512u : group);
                    keepAt      = lane * 8u + (row0 / 32u) % 2u * 4u;
                }
                else // (dword of block b, pair p, lane l: (((b / 2) * pairs + p) * 64 + l) * 2 + b % 2)
                    from[0] = static_cast<const char*>(scales) + ((static_cast<size_t>(row0 / 64u) * pairs * 64u + lane) * 2u + (row0 / 32u) % 2u) * 4u;
            }
            ROCWMMA_DEVICE ROCWMMA_INLINE void load(uint32_t(&to)[Raw ? 2u * Blocks : Blocks], uint32_t pair) const
            {
#pragma unroll
                for(uint32_t b = 0; b < Blocks; ++b)
                {
                    if constexpr(Raw)
                    {
                        typedef uint32_t Words __attribute__((ext_vector_type(2), aligned(4)));
                        const Words      v = *reinterpret_cast<const Words*>(from[b] + (8u * pair < last ? 8u * pair : last));
                        to[2u * b]         = v[0];
                        to[2u * b + 1u]    = v[1];
                    }
                    else
                        to[b] = reinterpret_cast<const uint32_t*>(from[0])[(static_cast<size_t>(b / 2u) * pairs + pair) * 128u + b % 2u];
                }
            }
            // The loaded pair `pair` takes over.
            ROCWMMA_DEVICE ROCWMMA_INLINE void take(uint32_t(&loaded)[Raw ? 2u * Blocks : Blocks], uint32_t pair)
            {
                const bool halfPair = 8u * pair > last; // (wave uniform)
#pragma unroll
                for(uint32_t b = 0; b < Blocks; ++b)
                {
                    if constexpr(Raw)
                    {
                        const uint32_t lo = halfPair ? loaded[2u * b + 1u] : loaded[2u * b], hi = halfPair ? 0x7f7f7f7fu : loaded[2u * b + 1u];
                        now[b]            = inside[b] ? packPairScales(lo, hi, lane) : 0x7f7f7f7fu;
                    }
                    else
                        now[b] = loaded[b];
                }
                if constexpr(Raw)
                {
                    // (a pair past the last lies past the end of the buffer as well)
                    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
                    if constexpr(Blocks == 2u)
                        __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{now[0], now[1]}, kept, static_cast<int>(keepAt + pair * 512u), 0, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b32(now[0], kept, static_cast<int>(keepAt + pair * 512u), 0, 0);
                }
            }
            // scale of block b at instruction step `step` (0..3) of the pair, in the lowest byte
            ROCWMMA_DEVICE ROCWMMA_INLINE uint32_t at(uint32_t b, uint32_t step) const
            {
                return now[b] >> (8u * step);
            }
        };

        // ---- stream-K support ------------------------------------------------------------------
        // Which part of a tile's K range a call of gemmTile computes.
        enum class TilePart
        {
            Whole, // all of K: the result goes through the epilogue
            Contributor, // a part that does not start at K = 0: the raw accumulators go to a workspace slot
            Owner // the part that starts at K = 0 of a tile other workgroups contribute to
        };

        // Workspace of the stream-K kernel: one slot of raw accumulators (MacroM x MacroN x 4 bytes, in
        // register order) and one flag per workgroup, then one word that records a wait that ran out
        // (kStreamKTimedOut; never cleared by a launch, only by the query that reports it) and the ticket
        // counter the workgroups of a launch draw their ranges from.
        constexpr uint32_t kStreamKTimedOut = 0x54494D45u; // "TIME": a value, not a bit, so that an uninitialised workspace does not read as a time-out
        struct StreamKPart
        {
            char*     slots; // slot i at slots + i * slotBytes
            uint32_t* flags; // flag i set to 1 once slot i is complete; [workgroups] = time-out marker, [workgroups + 1] = tickets
            uint32_t  slotBytes;
            uint32_t  mySlot; // contributor: where the accumulators go
            uint32_t  firstSlot, slotCount; // owner: the slots to add, in this order
            uint32_t  timeoutWord; // index of the time-out marker in flags
        };

        // Returns true when the caller is done with the tile (contributor).
        template <typename Cfg, TilePart Part, typename Acc>
        ROCWMMA_DEVICE ROCWMMA_INLINE bool streamKHandOver(Acc (&acc)[Cfg::BlocksM][Cfg::BlocksN], StreamKPart const& sk)
        {
            typedef uint32_t Words __attribute__((ext_vector_type(4)));
            constexpr uint32_t PerBlock = sizeof(acc[0][0].x) / 16u; // 16-byte pieces per accumulator block
            if constexpr(Part == TilePart::Contributor)
            {
                Words* slot = reinterpret_cast<Words*>(sk.slots + static_cast<size_t>(sk.mySlot) * sk.slotBytes);
#pragma unroll
                for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
#pragma unroll
                    for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
#pragma unroll
                        for(uint32_t p = 0; p < PerBlock; ++p)
                        {
                            Words v;
                            __builtin_memcpy(&v, reinterpret_cast<const char*>(acc[i][j].x) + 16u * p, 16);
                            slot[((i * Cfg::BlocksN + j) * PerBlock + p) * Cfg::Threads + threadIdx.x] = v;
                        }
                // Every thread's stores are visible device-wide before the flag is.  The barrier orders
                // the workgroup's stores before thread 0's releasing store, whose write-back of this L2
                // covers them all (the eight XCDs have an L2 each; one write-back per workgroup, not one
                // per wave: they are served one at a time and cost microseconds each).
                __syncthreads();
                if(threadIdx.x == 0u)
                    __hip_atomic_store(sk.flags + sk.mySlot, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                return true;
            }
            else
            {
                for(uint32_t c = 0; c < sk.slotCount; ++c)
                {
                    const uint32_t s = sk.firstSlot + c;
                    if(threadIdx.x == 0u)
                    {
                        // bounded wait: the contributors run their parts first, so the flag is normally
                        // up long before; a wait that runs out is recorded and the result is wrong
                        // rather than the device hung
                        // (relaxed polls: an acquiring load would invalidate this L2 on every poll and
                        // take the operand panels of the workgroups next door with it; the one fence
                        // that orders the slot reads follows below)
                        uint32_t spins = 0;
                        while(__hip_atomic_load(sk.flags + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u)
                        {
                            __builtin_amdgcn_s_sleep(8);
                            if(++spins > (1u << 22))
                            {
                                __hip_atomic_store(sk.flags + sk.timeoutWord, kStreamKTimedOut, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                break;
                            }
                        }
                        // one invalidation of this compute unit's L1 and this XCD's L2 for the workgroup
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                    }
                    __syncthreads();
                    const Words* slot = reinterpret_cast<const Words*>(sk.slots + static_cast<size_t>(s) * sk.slotBytes);
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
#pragma unroll
                        for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
#pragma unroll
                            for(uint32_t p = 0; p < PerBlock; ++p)
                            {
                                const Words v = slot[((i * Cfg::BlocksN + j) * PerBlock + p) * Cfg::Threads + threadIdx.x];
                                typename Cfg::CompT part[4];
                                __builtin_memcpy(part, &v, 16);
#pragma unroll
                                for(uint32_t e = 0; e < 4u; ++e)
                                    acc[i][j].x[4u * p + e] += part[e];
                            }
                    __syncthreads();
                    if(threadIdx.x == 0u) // taken: the next launch finds the flag down
                        __hip_atomic_store(sk.flags + s, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                return false;
            }
        }

        // Main loop schedules (per wave), by ring:
        //
        //   ring of two stages of 128 bytes of K (the 256 x 256 tile; N = 2 or 4 MFMA steps per stage), of three or with B a stage
        //   deeper (copies one stage further ahead, and left in flight at the wait):
        //     prologue : copies of stages 0 and 1 in flight; wait for stage 0; barrier; read F(0, step 0)
        //     stage i  : steps 0 .. N-2: read the next step's fragments while this step's MFMAs run
        //                wait: stage i+1 landed and own LDS reads returned;  barrier
        //                issue the copies of stage i+2 into stage i's slot, read F(i+1, step 0) while the
        //                  MFMAs of step N-1 run
        //     (fp8 16x16x128, one step per stage: the A fragments of a stage are held whole, the B fragments
        //     stream through column buffers; see that branch)
        //
        //   ring of S = 4 stages (64 or 128 bytes of K; F0 / F1 = fragment sets of a stage's two steps):
        //     prologue : copies for stages 0..2 in flight; wait for stage 0; barrier; read F0(0)
        //     stage i  : issue copies of stage i+3 (into the slot everybody finished reading at the
        //                  barrier of stage i-1); read F1(i) while the MFMAs of F0(i) run
        //                wait: stage i+1 landed (stages i+2, i+3 may stay in flight) and own LDS reads
        //                  returned;  barrier
        //                read F0(i+1) while the MFMAs of F1(i) run
        //
        // Every LDS read has a full MFMA step to return, and the barrier is the only synchronisation per
        // stage.
        // One macro tile (or, with Part != Whole, a part of its K range): tile (tm, tn) of the tile grid,
        // `stages` pipeline stages of K starting at stage `stage0`.
        // With an Emit other than Epilogue the results go to emit(acc, wave row, wave column) instead, once the LDS is free.
        struct Epilogue
        {
        };
        template <typename Cfg, TilePart Part = TilePart::Whole, typename Emit = Epilogue>
        ROCWMMA_DEVICE ROCWMMA_INLINE void gemmTile(uint32_t                   tm,
                                                    uint32_t                   tn,
                                                    uint32_t                   stage0,
                                                    uint32_t                   stages,
                                                    uint32_t                   m, // problem size: used by
                                                    uint32_t                   n, // configurations with edge
                                                    uint32_t                   k, // tiles only
                                                    typename Cfg::InT const*   a,
                                                    typename Cfg::InT const*   b,
                                                    typename Cfg::OutT const*  c,
                                                    typename Cfg::OutT*        d,
                                                    uint32_t                   lda,
                                                    uint32_t                   ldb,
                                                    uint32_t                   ldc,
                                                    uint32_t                   ldd,
                                                    typename Cfg::CompT        alpha,
                                                    typename Cfg::CompT        beta,
                                                    StreamKPart const&         sk,
                                                    TileExtras const&          ex = TileExtras{},
                                                    Emit const&                emit = Emit{})
        {
            const MxPacked& mx = ex.mx;
            using InT   = typename Cfg::InT;
            using OutT  = typename Cfg::OutT;
            using CompT = typename Cfg::CompT;
            using TileA = typename Cfg::TileA;
            using TileB = typename Cfg::TileB;

            extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];

            // (The thread index passes through an empty asm statement: in the persistent kernel, which
            // runs this function once per tile, everything derived from it would otherwise be hoisted
            // out of the tile loop and kept in registers across tiles, and the epilogue, which has none
            // to spare, would spill.)
            uint32_t tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            const uint32_t lane  = tid & 63u;
            const uint32_t wave  = __builtin_amdgcn_readfirstlane(tid >> 6); // wave uniform
            const uint32_t waveM = wave / Cfg::WavesN;
            const uint32_t waveN = wave % Cfg::WavesN;

            const uint32_t row0 = tm * Cfg::MacroM;
            const uint32_t col0 = tn * Cfg::MacroN;

            // Global sources: uniform tile pointer + uniform per-copy offset + per-lane offset
            const uint32_t ldaB = lda * sizeof(InT);
            const uint32_t ldbB = ldb * sizeof(InT);
            const char*    aSrc = reinterpret_cast<const char*>(a)
                               + static_cast<size_t>(row0) * (Cfg::AKMajor ? ldaB : static_cast<uint32_t>(sizeof(InT)));
            const char* bSrc = reinterpret_cast<const char*>(b)
                               + static_cast<size_t>(col0) * (Cfg::BKMajor ? ldbB : static_cast<uint32_t>(sizeof(InT)));
            // one past the last byte of each operand (edge tiles: the buffer bounds end there)
            const char* const aEnd = reinterpret_cast<const char*>(a)
                                     + (static_cast<size_t>((Cfg::AKMajor ? m : k) - 1u) * lda + (Cfg::AKMajor ? k : m)) * sizeof(InT);
            const char* const bEnd = reinterpret_cast<const char*>(b)
                                     + (static_cast<size_t>((Cfg::BKMajor ? n : k) - 1u) * ldb + (Cfg::BKMajor ? k : n)) * sizeof(InT);
            const size_t   aStep    = TileA::stageStep(ldaB);
            const size_t   bStep    = TileB::stageStep(ldbB);
            aSrc += aStep * stage0; // (the whole K range starts at stage 0)
            bSrc += bStep * stage0;
            // Issuers of the main loop's copies (Cfg::CopyWaves).  The partial tiles of the stream-K kernel keep
            // every wave issuing its own: with the issuer branch their instances, which already spill, ran
            // two to five times slower.
            constexpr uint32_t CopyWaves  = Part == TilePart::Whole ? Cfg::CopyWaves : Cfg::Waves;
            constexpr uint32_t CopyShares = Cfg::Waves / CopyWaves; // waves whose copies one issuer carries
            // (the lane offset of a copy depends on the wave it is issued for through the tile's swizzle: the
            // K-major tile's is the same for a wave and its partner, the dim-major tiles' are not)
            uint32_t aLaneOff[CopyShares], bLaneOff[CopyShares];
#pragma unroll
            for(uint32_t j = 0; j < CopyShares; ++j)
            {
                aLaneOff[j] = TileA::laneSourceOffset(lane, wave % CopyWaves + (Cfg::AKMajor ? 0u : j * CopyWaves), ldaB);
                bLaneOff[j] = TileB::laneSourceOffset(lane, wave % CopyWaves + (Cfg::BKMajor ? 0u : j * CopyWaves), ldbB);
            }

            // EdgesK: what is left of K (elements) at the stage the next copies read, and the first K element of
            // this lane's 16 bytes of a K-contiguous operand.  A lane whose bytes lie past the end of K asks for
            // an address beyond the buffer's bounds and gets zeros; rows of a dim-major operand past K are
            // beyond its end as they are.  Two vector instructions per operand and stage.
            uint32_t       aLeft = k - stage0 * Cfg::MacroK, bLeft = aLeft;
            const uint32_t aLaneK = TileA::laneK(lane, wave % CopyWaves) / static_cast<uint32_t>(sizeof(InT));
            const uint32_t bLaneK = TileB::laneK(lane, wave % CopyWaves) / static_cast<uint32_t>(sizeof(InT));
            auto           insideK = [](bool kMajor, uint32_t offset, uint32_t laneK, uint32_t left) {
                return (Cfg::EdgesK && kMajor && laneK >= left) ? (offset | 0x80000000u) : offset;
            };

            // A stage is copied in two halves (the A operand, then the B operand) so that each
            // MFMA phase of an iteration carries half of the copy instructions.
            // advance == false leaves the source on the stage just copied (used to re-copy the last
            // stage instead of running past the end of the operand; edge tiles read nothing there)
            auto issueA = [&](uint32_t slot, bool advance = true) {
                char*                 ldsA = ldsRaw + slot * Cfg::StrideA;
                const lds::BufferRsrc src  = Cfg::ScalarSources ? lds::makeScalarSource(aSrc, aEnd) : Cfg::Edges ? lds::makeSource(aSrc, aEnd) : lds::makeSource(aSrc);
                if constexpr(CopyWaves < Cfg::Waves)
                {
                    if(wave < CopyWaves)
                    {
#pragma unroll
                        for(uint32_t i = 0; i < Cfg::CopiesA * CopyShares; ++i)
                        {
                            // (copy i * CopyWaves + wave = copy i / CopyShares of wave + (i % CopyShares) * CopyWaves)
                            const uint32_t copy = i * CopyWaves + wave;
                            lds::asyncCopy16(ldsA + copy * 1024u, src, insideK(Cfg::AKMajor, aLaneOff[i % CopyShares], aLaneK, aLeft),
                                             TileA::copySourceOffset(copy, ldaB));
                        }
                    }
                }
                else
                {
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::CopiesA; ++i)
                    {
                        const uint32_t copy = i * Cfg::Waves + wave;
                        lds::asyncCopy16(ldsA + copy * 1024u, src, insideK(Cfg::AKMajor, aLaneOff[0], aLaneK, aLeft),
                                         TileA::copySourceOffset(copy, ldaB));
                    }
                }
                if constexpr(Cfg::EdgesK)
                {
                    aSrc += aStep;
                    aLeft = aLeft > Cfg::MacroK ? aLeft - Cfg::MacroK : 0u;
                }
                else
                    aSrc += advance ? aStep : size_t{0};
            };
            auto issueB = [&](uint32_t slot, bool advance = true) {
                char*                 ldsB = ldsRaw + Cfg::FirstB + slot * Cfg::StrideB;
                const lds::BufferRsrc src  = Cfg::ScalarSources ? lds::makeScalarSource(bSrc, bEnd) : Cfg::Edges ? lds::makeSource(bSrc, bEnd) : lds::makeSource(bSrc);
                if constexpr(CopyWaves < Cfg::Waves)
                {
                    if(wave < CopyWaves)
                    {
#pragma unroll
                        for(uint32_t i = 0; i < Cfg::CopiesB * CopyShares; ++i)
                        {
                            // (copy i * CopyWaves + wave = copy i / CopyShares of wave + (i % CopyShares) * CopyWaves)
                            const uint32_t copy = i * CopyWaves + wave;
                            lds::asyncCopy16(ldsB + copy * 1024u, src, insideK(Cfg::BKMajor, bLaneOff[i % CopyShares], bLaneK, bLeft),
                                             TileB::copySourceOffset(copy, ldbB));
                        }
                    }
                }
                else
                {
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::CopiesB; ++i)
                    {
                        const uint32_t copy = i * Cfg::Waves + wave;
                        lds::asyncCopy16(ldsB + copy * 1024u, src, insideK(Cfg::BKMajor, bLaneOff[0], bLaneK, bLeft),
                                         TileB::copySourceOffset(copy, ldbB));
                    }
                }
                if constexpr(Cfg::EdgesK)
                {
                    bSrc += bStep;
                    bLeft = bLeft > Cfg::MacroK ? bLeft - Cfg::MacroK : 0u;
                }
                else
                    bSrc += advance ? bStep : size_t{0};
            };
            auto issueStage = [&](uint32_t slot, bool advance = true) {
                issueA(slot, advance);
                issueB(slot, advance);
            };

            struct Frags
            {
                typename Cfg::FragA a[Cfg::BlocksM];
                typename Cfg::FragB b[Cfg::BlocksN];
            };

            auto readFragsOf = [&](Frags& f, uint32_t slot, uint32_t slotB, uint32_t ks) {
                const char* ldsA = ldsRaw + slot * Cfg::StrideA;
                const char* ldsB = ldsRaw + Cfg::FirstB + slotB * Cfg::StrideB;
                if constexpr(Cfg::Scaled && Cfg::Block == 16u) // (has a reader of its own in its loop)
                    return;
                else if constexpr(Cfg::Scaled)
                {
                    // 32x32x64 with block scales: the instruction's own K order, two runs of 16 bytes per lane from
                    // the two halves of the 64-byte step (chunks h and 2 + h of the step's four)
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
                    {
                        TileA::template readBlock32<16u>(f.a[i].x, ldsA, waveM * Cfg::WaveM + i * Cfg::Block, 2u * ks, lane);
                        TileA::template readBlock32<16u>(f.a[i].x + 16, ldsA, waveM * Cfg::WaveM + i * Cfg::Block, 2u * ks + 1u, lane);
                    }
#pragma unroll
                    for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
                    {
                        TileB::template readBlock32<16u>(f.b[j].x, ldsB, waveN * Cfg::WaveN + j * Cfg::Block, 2u * ks, lane);
                        TileB::template readBlock32<16u>(f.b[j].x + 16, ldsB, waveN * Cfg::WaveN + j * Cfg::Block, 2u * ks + 1u, lane);
                    }
                }
                else
                {
#pragma unroll
                for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
                {
                    if constexpr(Cfg::Block == 32u)
                        TileA::template readBlock32<Cfg::KPackBytes>(f.a[i].x, ldsA, waveM * Cfg::WaveM + i * Cfg::Block, ks, lane);
                    else
                        TileA::template readBlock16<Cfg::KPackBytes>(f.a[i].x, ldsA, waveM * Cfg::WaveM + i * Cfg::Block, ks, lane);
                }
#pragma unroll
                for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
                {
                    if constexpr(Cfg::Block == 32u)
                        TileB::template readBlock32<Cfg::KPackBytes>(f.b[j].x, ldsB, waveN * Cfg::WaveN + j * Cfg::Block, ks, lane);
                    else
                        TileB::template readBlock16<Cfg::KPackBytes>(f.b[j].x, ldsB, waveN * Cfg::WaveN + j * Cfg::Block, ks, lane);
                }
                }
            };

            auto readFrags = [&](Frags& f, uint32_t slot, uint32_t ks) { readFragsOf(f, slot, slot, ks); };

            // Fragments of a dim-major operand come from inline-assembly transposing reads: after the wait
            // that covers those reads, their registers are tied to that point of the program.
            auto pinFrags = [&](Frags& f) {
                if constexpr(!Cfg::AKMajor)
                {
#pragma unroll
                    for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
                        lds::pinRegisters(f.a[i].x);
                }
                if constexpr(!Cfg::BKMajor)
                {
#pragma unroll
                    for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
                        lds::pinRegisters(f.b[j].x);
                }
                (void)f;
            };

            typename Cfg::FragAcc acc[Cfg::BlocksM][Cfg::BlocksN];
#pragma unroll
            for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
#pragma unroll
                for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
                    fill_fragment(acc[i][j], static_cast<CompT>(0));

            auto multiply = [&](Frags const& f) {
#pragma unroll
                for(uint32_t i = 0; i < Cfg::BlocksM; ++i)
#pragma unroll
                    for(uint32_t j = 0; j < Cfg::BlocksN; ++j)
                        mma_sync(acc[i][j], f.a[i], f.b[j], acc[i][j]);
            };

            typename Cfg::FragC early[Cfg::PrefetchC ? Cfg::BlocksM : 1u][Cfg::PrefetchC ? Cfg::BlocksN : 1u];
            if constexpr(Cfg::PrefetchC)
            {
                if(beta != static_cast<CompT>(0))
                {
                    typedef uint32_t Words __attribute__((ext_vector_type(sizeof(OutT))));
                    const uint32_t   r0 = row0 + waveM * Cfg::WaveM + (lane & (Cfg::Block - 1u)), c0 = col0 + waveN * Cfg::WaveN + 4u * (lane / Cfg::Block);
#pragma unroll
                    for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t r = 0; r < Cfg::FragC::num_elements / 4u; ++r)
                            {
                                const uint32_t row = r0 + bi * Cfg::Block, col = c0 + bj * Cfg::Block + 8u * r;
                                Words          v   = {};
                                if(!Cfg::Edges || (row < m && col < n))
                                    v = *reinterpret_cast<const Words*>(c + static_cast<size_t>(row) * ldc + col);
                                __builtin_memcpy(early[bi][bj].x + 4u * r, &v, sizeof(v));
                            }
                }
                __builtin_amdgcn_sched_barrier(0);
            }

            // Where a wave's rows begin in the tile, and the row of its block bi behind that.  Wide waves: 128 rows, or, where rows of a 32-bit D are
            // a multiple of 32 KiB apart, two runs of 64, in turn with the other waves' runs.  The waves write the same block of theirs at about
            // the same time, and with 128 rows between them that is 4 MiB, which the memory channels do not tell apart; nor do they 1 MiB, which
            // is why runs of 64 rows are not taken for rows of 16 KiB.  bf16, eight waves of 64 x 128, runs of 128, of 64: with C 4096 x 8192 x 256
            // 61.4, 75.0, 62.0 us, x 1024 92.3, 102.1, 91.2; 8192 x 4096 x 256 69.0, 61.0, 70.1, x 1024 99.4, 90.2, 98.1; without C 8192 x 8192 x 256
            // 72.0, 77.9, 69.7.  (16-bit D, 4096 x 16384 x 1024 with C 156.8, 140.6, 145.9.)
            constexpr bool RunsOfD  = Cfg::WideWave && sizeof(OutT) == 4u;
            const bool     twoRuns  = RunsOfD && static_cast<uint32_t>(ldd * sizeof(OutT)) % 32768u == 0u;
            const uint32_t waveRow  = waveM * (twoRuns ? Cfg::WaveM / 2u : Cfg::WaveM);
            const uint32_t upperRow = twoRuns ? Cfg::MacroM / 2u : Cfg::WaveM / 2u;
            auto           blockRow = [&](uint32_t bi) {
                if constexpr(RunsOfD)
                    return bi < Cfg::BlocksM / 2u ? bi * Cfg::Block : upperRow + (bi - Cfg::BlocksM / 2u) * Cfg::Block;
                else
                    return bi * Cfg::Block;
            };

            // Wide waves: the accumulators while they are summed.  The epilogue takes them a row of blocks at a time (takeRow), so that
            // only that row is in ordinary registers: row bi of blocks to acc[at].
            typedef CompT Result __attribute__((ext_vector_type(4)));
            Result        sum[Cfg::WideWave ? Cfg::BlocksM : 1u][Cfg::WideWave ? Cfg::BlocksN : 1u];
            auto          takeRow = [&](uint32_t bi, uint32_t at) {
                if constexpr(Cfg::RolledRows)
                {
                    // (which row is known when the kernel runs: a branch per row around the moves out of the accumulation registers, which are
                    // written in assembly because the compiler makes them in front of the loop else, for all rows, and spills)
#pragma unroll
                    for(uint32_t r = 0; r < Cfg::BlocksM; ++r)
                        if(bi == r)
                        {
#pragma unroll
                            for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                                for(uint32_t e = 0; e < 4u; ++e)
                                {
                                    const CompT from = sum[r][bj][e];
                                    CompT       to;
#if ROCWMMA_ARCH_GFX950
                                    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(to) : "a"(from));
#else
                                    to = from;
#endif
                                    acc[at][bj].x[e] = to;
                                }
                        }
                }
                else if constexpr(Cfg::WideWave)
                {
#pragma unroll
                    for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                    {
                        asm volatile("" : "+a"(sum[bi][bj]));
#pragma unroll
                        for(uint32_t e = 0; e < 4u; ++e)
                            acc[at][bj].x[e] = sum[bi][bj][e];
                    }
                }
                (void)bi, (void)at;
            };

            constexpr uint32_t S      = Cfg::Stages;
            // `stages` stages of K from stage0 on: >= S - 1 of them (checked by the host)

            if constexpr(Cfg::WideWave)
            {
                // Four waves of 128 x 128 (128 x 64 in half tiles), one per SIMD; A ring of two stages of 128 bytes, B ring of three (256 x 128
                // tiles: three and four).
                // Against eight waves of 64 x 128 every LDS byte feeds a third more flops, nothing is issued twice and the copies are
                // spread over the whole stage: those of B(i + S) over its first step, those of A(i + S) over the second, one to eight
                // matrix instructions, so no wave ever queues behind them.  What bounds it is the power cap: 2290 clocks a stage
                // without reads and copies, 2420 with (2048 of matrix work), 1.7 GHz on normally distributed data, 2.4 on zeros.
                // 8192^3: bf16 both row-major 840 -> 780 us, f16 A row-major / B col-major 807 -> 762; 4096^3 112.7 -> 105.7, 109 -> 101.6.
                // The matrix instructions are written in assembly: with the builtins the compiler moves all accumulators through
                // ordinary registers once per stage (twice the time).  They go through the blocks in squares of 2 x 2, along and back, so
                // that each shares an operand with the one before (row by row: 1.0-1.5 % slower under the power cap).
                static_assert(Part == TilePart::Whole && std::is_same<Emit, Epilogue>::value && !Cfg::PrefetchC && Cfg::KSteps == 2u && Cfg::KPackBytes == 16u && Cfg::BlocksN % 2u == 0u, "wide waves: whole K ranges, two steps a stage");
                constexpr uint32_t TurnsA = Cfg::TurnsA, TurnsB = Cfg::TurnsB;
                uint32_t           aOff[TurnsA], bOff[TurnsB];
#pragma unroll
                for(uint32_t t = 0; t < TurnsA; ++t)
                    aOff[t] = TileA::laneSourceOffset(lane, wave + t * Cfg::Waves, ldaB);
#pragma unroll
                for(uint32_t t = 0; t < TurnsB; ++t)
                    bOff[t] = TileB::laneSourceOffset(lane, wave + t * Cfg::Waves, ldbB);
                auto sourceA = [&] { return Cfg::Edges ? lds::makeSource(aSrc, aEnd) : lds::makeSource(aSrc); };
                auto sourceB = [&] { return Cfg::Edges ? lds::makeSource(bSrc, bEnd) : lds::makeSource(bSrc); };
                auto copyA = [&](uint32_t slot, uint32_t i, lds::BufferRsrc const& src) {
                    const uint32_t copy = i * Cfg::Waves + wave;
                    lds::asyncCopy16(ldsRaw + slot * Cfg::StrideA + copy * 1024u, src, insideK(Cfg::AKMajor, aOff[i % TurnsA], aLaneK, aLeft),
                                     TileA::copySourceOffset(copy, ldaB));
                };
                auto copyB = [&](uint32_t slot, uint32_t i, lds::BufferRsrc const& src) {
                    const uint32_t copy = i * Cfg::Waves + wave;
                    lds::asyncCopy16(ldsRaw + Cfg::FirstB + slot * Cfg::StrideB + copy * 1024u, src, insideK(Cfg::BKMajor, bOff[i % TurnsB], bLaneK, bLeft),
                                     TileB::copySourceOffset(copy, ldbB));
                };
                // (more == false: the last stage is copied again, into a slot nobody reads; edge tiles read nothing there)
                auto advanceA = [&](bool more) {
                    aSrc += Cfg::EdgesK || more ? aStep : size_t{0};
                    if constexpr(Cfg::EdgesK)
                        aLeft = aLeft > Cfg::MacroK ? aLeft - Cfg::MacroK : 0u;
                };
                auto advanceB = [&](bool more) {
                    bSrc += Cfg::EdgesK || more ? bStep : size_t{0};
                    if constexpr(Cfg::EdgesK)
                        bLeft = bLeft > Cfg::MacroK ? bLeft - Cfg::MacroK : 0u;
                };
                typedef uint32_t Operand __attribute__((ext_vector_type(4)));
                Operand          fa[2][Cfg::BlocksM], fb[2][Cfg::BlocksN];
#pragma unroll
                for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
#pragma unroll
                    for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                        sum[bi][bj] = Result{0, 0, 0, 0};
                constexpr uint32_t Reads = Cfg::BlocksM + Cfg::BlocksN, Mfmas = Cfg::BlocksM * Cfg::BlocksN;
                // operand q of a step: the blocks of A, then those of B
                auto readOperand = [&](uint32_t set, uint32_t slotA, uint32_t slotB, uint32_t ks, uint32_t q) {
                    if(q < Cfg::BlocksM)
                        TileA::template readBlock16<16u>(&fa[set][q], ldsRaw + slotA * Cfg::StrideA, waveRow + blockRow(q), ks, lane);
                    else
                        TileB::template readBlock16<16u>(&fb[set][q - Cfg::BlocksM], ldsRaw + Cfg::FirstB + slotB * Cfg::StrideB,
                                                         waveN * Cfg::WaveN + (q - Cfg::BlocksM) * 16u, ks, lane);
                };
                auto pinSet = [&](uint32_t set) {
#pragma unroll
                    for(uint32_t q = 0; q < Cfg::BlocksM; ++q)
                        lds::pinRegisters(fa[set][q]);
#pragma unroll
                    for(uint32_t q = 0; q < Cfg::BlocksN; ++q)
                        lds::pinRegisters(fb[set][q]);
                };
                // (the accumulators are kept transposed: the instruction's first multiplicand is B)
                auto multiplyBlock = [&](uint32_t set, uint32_t bi, uint32_t bj) {
#if ROCWMMA_ARCH_GFX950
                    if constexpr(std::is_same<InT, float16_t>::value)
                        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(sum[bi][bj]) : "v"(fb[set][bj]), "v"(fa[set][bi]));
                    else if constexpr(sizeof(InT) == 2u)
                        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(sum[bi][bj]) : "v"(fb[set][bj]), "v"(fa[set][bi]));
                    else
                        asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(sum[bi][bj]) : "v"(fb[set][bj]), "v"(fa[set][bi]));
#else
                    (void)set, (void)bi, (void)bj;
#endif
                };
                // One step on fragment set `set`: its matrix instructions, the next step's reads among the first three quarters of them and
                // `Copies` copies spread over all.
                auto step = [&](auto setC, auto&& read, auto copiesC, auto&& copy) {
                    constexpr uint32_t set = decltype(setC)::value, Copies = decltype(copiesC)::value;
                    constexpr uint32_t PerRead = Mfmas * 3u / 4u / Reads, PerCopy = Mfmas / Copies, Squares = Cfg::BlocksN / 2u;
#pragma unroll
                    for(uint32_t x = 0; x < Mfmas; ++x)
                    {
                        const uint32_t square = x / 4u, inside = x % 4u, si = square / Squares;
                        const uint32_t sj     = si % 2u == 0u ? square % Squares : Squares - 1u - square % Squares;
                        multiplyBlock(set, 2u * si + inside / 2u, 2u * sj + ((inside / 2u) ^ (inside % 2u)));
                        const bool readNow = x % PerRead == 0u && x / PerRead < Reads, copyNow = x % PerCopy == PerCopy / 2u && x / PerCopy < Copies;
                        if(readNow)
                            read(x / PerRead);
                        if(copyNow)
                            copy(x / PerCopy);
                        if(readNow || copyNow)
                            __builtin_amdgcn_sched_barrier(0);
                    }
                };
#pragma unroll
                for(uint32_t st = 0; st < S; ++st)
                {
                    const lds::BufferRsrc srcA = sourceA(), srcB = sourceB();
#pragma unroll
                    for(uint32_t c = 0; c < Cfg::CopiesA; ++c)
                        copyA(st, c, srcA);
#pragma unroll
                    for(uint32_t c = 0; c < Cfg::CopiesB; ++c)
                        copyB(st, c, srcB);
                    advanceA(st + 1u < stages);
                    advanceB(st + 1u < stages);
                }
                lds::waitCopiesAndReads<(S - 1u) * Cfg::Copies>(); // stage 0 has landed
                lds::barrier();
#pragma unroll
                for(uint32_t q = 0; q < Reads; ++q)
                    readOperand(0u, 0u, 0u, 0u, q);
                lds::waitReads();
                pinSet(0u);
                // (slots of stage i; the slot of B that stage i - 1 has left is the one that is in front of stage i's)
                uint32_t slotA = 0u, slotB = 0u, freeB = S;
                for(uint32_t i = 0; i < stages; ++i)
                {
                    const uint32_t nextA = slotA == S - 1u ? 0u : slotA + 1u, nextB = slotB == S ? 0u : slotB + 1u;
                    __builtin_amdgcn_sched_barrier(0);
                    const lds::BufferRsrc srcB = sourceB();
                    step(std::integral_constant<uint32_t, 0u>{}, [&](uint32_t q) { readOperand(1u, slotA, slotB, 1u, q); },
                         std::integral_constant<uint32_t, Cfg::CopiesB>{}, [&](uint32_t c) { copyB(freeB, c, srcB); });
                    advanceB(i + S + 1u < stages);
                    __builtin_amdgcn_sched_barrier(0);
                    // stage i + 1 has landed (the stages behind it and B of stage i + S may be in flight), stage i is in registers
                    lds::waitCopiesAndReads<(S - 2u) * Cfg::Copies + Cfg::CopiesB>();
                    pinSet(1u);
                    lds::barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    const lds::BufferRsrc srcA = sourceA();
                    step(std::integral_constant<uint32_t, 1u>{}, [&](uint32_t q) { readOperand(0u, nextA, nextB, 0u, q); },
                         std::integral_constant<uint32_t, Cfg::CopiesA>{}, [&](uint32_t c) { copyA(slotA, c, srcA); });
                    advanceA(i + S + 1u < stages);
                    freeB = slotB;
                    slotA = nextA;
                    slotB = nextB;
                    __builtin_amdgcn_sched_barrier(0);
                    lds::waitReads();
                    pinSet(0u);
                }
                lds::waitCopiesAndReads<0u>(); // the surplus copies still target this workgroup's LDS
                lds::barrier();
                // (the compiler does not know the last matrix instructions: their results are written 16 clocks or so behind them)
                asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
            }
            else if constexpr(S == 2u && Cfg::KSteps == 1u)
            {
                // Ring of two stages, one MFMA step per stage whose fragments would not fit the register
                // file twice (fp8 16x16x128: 8 registers per block and operand).  The A fragments of a
                // stage are held whole (and read one stage ahead into a second set); the B fragments
                // stream through column buffers: while column j is multiplied, column j + Ahead is read.
                // The barrier sits in front of the last Ahead columns: by then the wave has read everything
                // it needs from stage i (the last columns' fragments arrived with the wait), stage i + 1 has
                // landed, and the copies of stage i + 2 go out into stage i's slot.
                static_assert(Cfg::AKMajor && Cfg::BKMajor, "streamed columns: K-contiguous operands");
                static_assert(!Cfg::Scaled || Part == TilePart::Whole, "block scales: whole K ranges from stage 0");
                // Block scales (Scaled only): per lane, pair of stages and group of four blocks, two
                // registers: byte (block % 2) * 2 + stage parity of register (block % 4) / 2.  The next
                // pair's are loaded while the first stage of a pair is multiplied and take over after the
                // second.
                typedef uint32_t   Scales __attribute__((ext_vector_type(2)));
                constexpr uint32_t GroupsN = Cfg::BlocksN / 4u;
                static_assert(!Cfg::Scaled || (Cfg::BlocksM == 4u && Cfg::BlocksN % 4u == 0u), "packed scales: groups of four blocks");
                Scales        sA = {}, sAnext = {};
                Scales        sB[GroupsN > 0u ? GroupsN : 1u] = {}, sBnext[GroupsN > 0u ? GroupsN : 1u] = {};
                const Scales* mxA = nullptr;
                const Scales* mxB = nullptr;
                auto loadScales = [&](Scales& a_, Scales(&b_)[GroupsN > 0u ? GroupsN : 1u], uint32_t pair) {
                    a_ = mxA[static_cast<size_t>(pair) * 64u];
#pragma unroll
                    for(uint32_t gN = 0; gN < GroupsN; ++gN)
                        b_[gN] = mxB[(static_cast<size_t>(gN) * mx.pairs + pair) * 64u];
                };
                if constexpr(Cfg::Scaled)
                {
                    mxA = static_cast<const Scales*>(mx.a) + static_cast<size_t>(row0 / 64u + waveM) * mx.pairs * 64u + lane;
                    mxB = static_cast<const Scales*>(mx.b) + static_cast<size_t>(col0 / 64u + waveN * GroupsN) * mx.pairs * 64u + lane;
                    // (in front of the first copies: the wait for stage 0 below then covers these loads, and the
                    // loop is entered with none of them in flight)
                    loadScales(sA, sB, 0u);
                    __builtin_amdgcn_sched_barrier(0); // (and stay in front of them)
                }
                constexpr uint32_t SB = Cfg::StagesB;
#pragma unroll
                for(uint32_t st = 0; st < SB; ++st)
                {
                    if(st < S)
                        issueA(st, st + 1u < stages);
                    issueB(st, st + 1u < stages);
                }
                constexpr uint32_t InFlight = (SB - 2u) * Cfg::CopiesB * CopyShares;
                lds::waitCopiesAndReads<(Cfg::CopiesA + (SB - 1u) * Cfg::CopiesB) * CopyShares>(); // stage 0 has landed
                lds::barrier();
                uint32_t slotB = 0u; // of the stage that is multiplied
                // B column buffers: `Ahead` columns are read in advance.  With three (four buffers, whose indices
                // repeat every stage of four or eight columns) the barrier moves in front of the last three
                // columns, so that what follows it (the copies, the next stage's A fragments and first B columns)
                // has twelve MFMAs to hide behind instead of four: 252 registers, no spills, fp8
                // 4096 x 14336 x 4096 194.0 -> 190.3 us.  The kernel with block scales keeps one column ahead
                // (its scale registers take the room).
                constexpr uint32_t Ahead = (!Cfg::Scaled && Cfg::BlocksN % 4u == 0u) ? 3u : 1u;
                constexpr uint32_t NB    = Ahead + 1u;
                static_assert(Cfg::BlocksN % NB == 0u && Cfg::BlocksN > Ahead, "the buffer of a column must not depend on the stage");
                typename Cfg::FragA fa[2][Cfg::BlocksM];
                typename Cfg::FragB fb[NB];
                auto readA = [&](typename Cfg::FragA(&dst)[Cfg::BlocksM], uint32_t slot) {
                    const char* ldsA = ldsRaw + slot * Cfg::StrideA;
#pragma unroll
                    for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                    {
                        const uint32_t r0 = waveM * Cfg::WaveM + bi * Cfg::Block;
                        if constexpr(Cfg::Scaled)
                        {
                            TileA::template readBlock16<16u>(dst[bi].x, ldsA, r0, 0u, lane);
                            TileA::template readBlock16<16u>(dst[bi].x + 16, ldsA, r0, 1u, lane);
                        }
                        else
                            TileA::template readBlock16<Cfg::KPackBytes>(dst[bi].x, ldsA, r0, 0u, lane);
                    }
                };
                auto readB = [&](typename Cfg::FragB& dst, uint32_t slot, uint32_t bj) {
                    const char*    ldsB = ldsRaw + Cfg::FirstB + slot * Cfg::StrideB;
                    const uint32_t c0   = waveN * Cfg::WaveN + bj * Cfg::Block;
                    if constexpr(Cfg::Scaled)
                    {
                        TileB::template readBlock16<16u>(dst.x, ldsB, c0, 0u, lane);
                        TileB::template readBlock16<16u>(dst.x + 16, ldsB, c0, 1u, lane);
                    }
                    else
                        TileB::template readBlock16<Cfg::KPackBytes>(dst.x, ldsB, c0, 0u, lane);
                };
                auto column = [&](typename Cfg::FragA const(&a_)[Cfg::BlocksM], typename Cfg::FragB const& b_, auto bjC, auto stC) {
                    constexpr uint32_t bj = decltype(bjC)::value, st = decltype(stC)::value;
                    if constexpr(Cfg::Scaled)
                    {
#if ROCWMMA_ARCH_GFX950 // (the instruction table exists in the device pass only)
                        using Op  = detail::MfmaScaled<detail::TypeInfo<InT>::cls, detail::TypeInfo<InT>::cls, 16u>;
                        using Acc = typename Op::Acc;
                        staticFor<Cfg::BlocksM>([&](auto biC) {
                            constexpr uint32_t bi = decltype(biC)::value;
                            Acc&               v  = *reinterpret_cast<Acc*>(acc[bi][bj].x);
                            // (the accumulator is kept transposed: the instruction's first multiplicand is B)
                            v = Op::template exec<(bj % 2u) * 2u + st, (bi % 2u) * 2u + st>(b_.x, a_[bi].x, v, sB[bj / 4u][(bj % 4u) / 2u],
                                                                                           sA[bi / 2u]);
                        });
#else
                        (void)a_, (void)b_, (void)bj, (void)st;
#endif
                    }
                    else
                    {
#pragma unroll
                        for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                            mma_sync(acc[bi][bj], a_[bi], b_, acc[bi][bj]);
                    }
                };
                constexpr uint32_t RB = Cfg::KPackBytes / 16u; // LDS reads per block
                readA(fa[0], 0u);
#pragma unroll
                for(uint32_t j = 0; j < Ahead; ++j)
                    readB(fb[j], 0u, j);
                // (the A sets alternate with the stage parity; two stages per trip keep the indices static)
                auto stage = [&](typename Cfg::FragA(&cur)[Cfg::BlocksM], typename Cfg::FragA(&nxt)[Cfg::BlocksM], auto slotC,
                                 uint32_t ii) {
                        constexpr uint32_t slot = decltype(slotC)::value;
                        staticFor<Cfg::BlocksN - Ahead>([&](auto bjC) {
                            constexpr uint32_t bj = decltype(bjC)::value;
                            readB(fb[(bj + Ahead) % NB], slotB, bj + Ahead);
                            column(cur, fb[bj % NB], bjC, slotC);
                            scheduleInterleaved<Cfg::BlocksM, RB, 0u>();
                            __builtin_amdgcn_sched_barrier(0);
                        });
                        lds::waitCopiesAndReads<InFlight>(); // stage ii + 1 has landed, stage ii is in registers
                        lds::barrier();
                        __builtin_amdgcn_sched_barrier(0);
                        issueA(slot, ii + 3u < stages);
                        issueB(slotB, ii + SB + 1u < stages);
                        slotB = slotB + 1u == SB ? 0u : slotB + 1u;
                        if constexpr(Cfg::Scaled && slot == 0u)
                        {
                            // scales of the next pair of stages (the last pair again past the end of K)
                            loadScales(sAnext, sBnext, ii / 2u + 1u < mx.pairs ? ii / 2u + 1u : mx.pairs - 1u);
                        }
                        readA(nxt, slot ^ 1u);
                        staticFor<Ahead>([&](auto tC) {
                            constexpr uint32_t t  = decltype(tC)::value;
                            constexpr uint32_t bj = Cfg::BlocksN - Ahead + t;
                            readB(fb[(bj + Ahead) % NB], slotB, t);
                            column(cur, fb[bj % NB], std::integral_constant<uint32_t, bj>{}, slotC);
                            if constexpr(Ahead > 1u)
                                __builtin_amdgcn_sched_barrier(0);
                        });
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr(Cfg::Scaled && slot == 1u)
                        {
                            sA = sAnext;
#pragma unroll
                            for(uint32_t gN = 0; gN < GroupsN; ++gN)
                                sB[gN] = sBnext[gN];
                        }
                };
                const std::integral_constant<uint32_t, 0u> even{};
                const std::integral_constant<uint32_t, 1u> odd{};
                uint32_t i = 0;
                for(; i + 1u < stages; i += 2u)
                {
                    stage(fa[0], fa[1], even, i);
                    stage(fa[1], fa[0], odd, i + 1u);
                }
                if(i < stages)
                    stage(fa[0], fa[1], even, i);
                lds::waitCopiesAndReads<0u>(); // the surplus copies still target this workgroup's LDS
                lds::barrier();
            }
            else if constexpr(S == 2u || S == 3u)
            {
                // Ring of two or three stages of 128 bytes of K (two or four MFMA steps each), the ring of B perhaps a stage
                // deeper.  A phase multiplies
                // one step while it reads the fragments of the next; the barrier in front of a stage's
                // last phase is where stage i has been read completely and stage i+1 has landed, so
                // the copies of stage i+2 go out right behind it, into stage i's slot, and have the
                // phases up to the next barrier to land.  Past the end of K the loop copies the
                // last stage again and reads fragments nobody multiplies, so its body is uniform.
                // Block scales (Scaled, 32-wide blocks): per lane and pair of stages (256 bytes of K = four
                // instruction steps), one dword per block of 32 rows, byte = step; the step's byte is shifted
                // down at run time.  The next pair's are loaded behind the barrier of a pair's first stage.
                static_assert(!Cfg::Scaled || Cfg::KSteps == 2u, "packed scales: two instruction steps per stage");
                PairScales<Cfg, Cfg::Scaled ? Cfg::BlocksM : 1u> sA(mx.a, mx.lda, mx.pairs, row0 + waveM * Cfg::WaveM, m, k, lane, mx.packedA, tn == 0u && waveN == 0u);
                PairScales<Cfg, Cfg::Scaled ? Cfg::BlocksN : 1u> sB(mx.b, mx.ldb, mx.pairs, col0 + waveN * Cfg::WaveN, n, k, lane, mx.packedB, tm == 0u && waveM == 0u);
                if constexpr(Cfg::Scaled)
                {
                    // (in front of the first copies and kept there: the wait for stage 0 then covers these loads,
                    // and the loop is entered with none of them in flight)
                    sA.load(sA.next, 0u);
                    sB.load(sB.next, 0u);
                    __builtin_amdgcn_sched_barrier(0);
                }
                constexpr uint32_t SB = Cfg::StagesB;
#pragma unroll
                for(uint32_t st = 0; st < SB; ++st)
                {
                    if(st < S)
                        issueA(st, st + 1u < stages);
                    issueB(st, st + 1u < stages);
                }
                if constexpr(Cfg::Scaled)
                {
                    __builtin_amdgcn_sched_barrier(0);
                    sA.take(sA.next, 0u);
                    sB.take(sB.next, 0u);
                }
                // (copies of later stages that may be in flight when a stage must have landed; the waves that issue
                // none do not wait)
                constexpr uint32_t InFlight = ((S - 2u) * Cfg::CopiesA + (SB - 2u) * Cfg::CopiesB) * CopyShares;
                lds::waitCopiesAndReads<((S - 1u) * Cfg::CopiesA + (SB - 1u) * Cfg::CopiesB) * CopyShares>(); // stage 0 has landed
                lds::barrier();
                constexpr uint32_t N = Cfg::KSteps; // MFMA steps per stage: 2 or 4 (even: the fragment sets alternate)
                Frags              f[2];
                auto multiplyStep = [&](Frags const& fr, uint32_t i, uint32_t ks) {
                    if constexpr(Cfg::Scaled)
                    {
#if ROCWMMA_ARCH_GFX950 // (the instruction table exists in the device pass only)
                        using Op  = detail::MfmaScaled<detail::TypeInfo<InT>::cls, detail::TypeInfo<InT>::cls, 32u>;
                        using Acc = typename Op::Acc;
                        const uint32_t step = (i % 2u) * N + ks; // within the pair of stages
#pragma unroll
                        for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
#pragma unroll
                            for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                            {
                                Acc& v = *reinterpret_cast<Acc*>(acc[bi][bj].x);
                                // (the accumulator is kept transposed: the instruction's first multiplicand is B)
                                v = Op::template exec<0, 0>(fr.b[bj].x, fr.a[bi].x, v, sB.at(bj, step), sA.at(bi, step));
                            }
#else
                        (void)fr, (void)i, (void)ks;
#endif
                    }
                    else
                    {
                        (void)i, (void)ks;
                        multiply(fr);
                    }
                };
                readFrags(f[0], 0u, 0u);
                // Slots of stage i.  Rings of two: its parity, taken where it is needed.  (Held in a variable over the body, the
                // LDS addresses made from it stayed live with it: the stream-K kernels spilled 245 to 360 registers instead of 160
                // to 256, 2560 x 2560 x 8192 int8 115.8 -> 131.9 us.)
                constexpr bool ParityA = S == 2u, ParityB = SB == 2u;
                uint32_t       ringA = 0u, ringB = 0u;
                auto           slotA = [&](uint32_t i) { return ParityA ? i % 2u : ringA; };
                auto           slotB = [&](uint32_t i) { return ParityB ? i % 2u : (SB == S ? slotA(i) : ringB); };
                for(uint32_t i = 0; i < stages; ++i)
                {
#pragma unroll
                    for(uint32_t ks = 0; ks + 1u < N; ++ks)
                    {
                        if constexpr(!Cfg::AKMajor || !Cfg::BKMajor)
                        {
                            lds::waitReads(); // transposing reads of the previous phase
                            pinFrags(f[ks & 1u]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        readFragsOf(f[(ks + 1u) & 1u], slotA(i), slotB(i), ks + 1u);
                        multiplyStep(f[ks & 1u], i, ks);
                        scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    lds::waitCopiesAndReads<InFlight>(); // stage i+1 has landed, stage i is in registers
                    pinFrags(f[(N - 1u) & 1u]);
                    lds::barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    issueA(slotA(i), i + S + 1u < stages);
                    issueB(slotB(i), i + SB + 1u < stages);
                    if constexpr(Cfg::Scaled)
                    {
                        if(i % 2u == 0u)
                        {
                            sA.load(sA.next, i / 2u + 1u < mx.pairs ? i / 2u + 1u : mx.pairs - 1u);
                            sB.load(sB.next, i / 2u + 1u < mx.pairs ? i / 2u + 1u : mx.pairs - 1u);
                        }
                    }
                    if constexpr(!ParityA)
                        ringA = ringA + 1u == S ? 0u : ringA + 1u;
                    if constexpr(SB != S)
                        ringB = ringB + 1u == SB ? 0u : ringB + 1u;
                    readFragsOf(f[0], slotA(i + 1u), slotB(i + 1u), 0u);
                    multiplyStep(f[(N - 1u) & 1u], i, N - 1u);
                    if constexpr(Cfg::Scaled)
                    {
                        if(i % 2u == 1u)
                        {
                            sA.take(sA.next, i / 2u + 1u);
                            sB.take(sB.next, i / 2u + 1u);
                        }
                    }
                    scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                    scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::Copies>();
                    __builtin_amdgcn_sched_barrier(0);
                }
                lds::waitCopiesAndReads<0u>(); // the surplus copies still target this workgroup's LDS
                lds::barrier();
            }
            else if constexpr(Cfg::KSteps == 2u && Cfg::Scaled)
            {
                // Ring of four stages of 128 bytes of K with block scales (32-wide blocks, two instruction steps per
                // stage): the loop below with the scale loads joining its count of vector-memory operations in
                // flight.  Two stages per trip, so that a trip is one pair of stages of the packed scales (one dword
                // per block and lane, byte = step of the pair) and everything that depends on a stage's parity is a
                // constant: the next pair's scales are requested at the head of a trip, two stages before they take
                // over.  Every trip issues its stages (past the end of K the last stage again, into a slot nobody
                // reads), so the body and its counts are uniform.
                static_assert(S == 4u && Cfg::StageKB == 128u && Cfg::Block == 32u && Part == TilePart::Whole, "scaled ring of four: 128-byte stages of 32-wide blocks");
                PairScales<Cfg, Cfg::BlocksM> sA(mx.a, mx.lda, mx.pairs, row0 + waveM * Cfg::WaveM, m, k, lane, mx.packedA, tn == 0u && waveN == 0u);
                PairScales<Cfg, Cfg::BlocksN> sB(mx.b, mx.ldb, mx.pairs, col0 + waveN * Cfg::WaveN, n, k, lane, mx.packedB, tm == 0u && waveM == 0u);
                auto multiplyScaled = [&](Frags const& fr, auto stepC) {
#if ROCWMMA_ARCH_GFX950 // (the instruction table exists in the device pass only)
                    using Op  = detail::MfmaScaled<detail::TypeInfo<InT>::cls, detail::TypeInfo<InT>::cls, 32u>;
                    using Acc = typename Op::Acc;
                    constexpr uint32_t step = decltype(stepC)::value; // within the pair of stages
#pragma unroll
                    for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                        {
                            Acc& v = *reinterpret_cast<Acc*>(acc[bi][bj].x);
                            // (the accumulator is kept transposed: the instruction's first multiplicand is B)
                            v = Op::template exec<0, 0>(fr.b[bj].x, fr.a[bi].x, v, sB.at(bj, step), sA.at(bi, step));
                        }
#else
                    (void)fr, (void)stepC;
#endif
                };
                // (in front of the first copies and kept there: the wait for stage 0 covers them)
                sA.load(sA.next, 0u);
                sB.load(sB.next, 0u);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for(uint32_t st = 0; st < S - 1u; ++st)
                    issueStage(st, st + 1u < stages);
                __builtin_amdgcn_sched_barrier(0);
                sA.take(sA.next, 0u);
                sB.take(sB.next, 0u);
                lds::waitCopiesAndReads<(S - 2u) * Cfg::Copies>();
                lds::barrier();
                Frags f0, f1;
                readFrags(f0, 0u, 0u);
                auto stage = [&](uint32_t i, auto parityC) {
                    constexpr uint32_t parity = decltype(parityC)::value;
                    const uint32_t     slot   = (i + S - 1u) % S;
                    const bool         adv    = i + S < stages;
                    issueA(slot, adv);
                    readFrags(f1, i % S, 1u);
                    multiplyScaled(f0, std::integral_constant<uint32_t, parity * 2u>{});
                    scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                    scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::CopiesA>();
                    __builtin_amdgcn_sched_barrier(0);
                    // Stage i+1 has landed once only stage i+2 and the A half of stage i+3 are in flight.  The scale
                    // loads of a trip's head sit between those two in issue order, but loads into registers do not
                    // complete in order with copies into LDS (counting them as in flight let a wait pass with a copy of
                    // stage i+1 outstanding whenever they had returned first: wrong results on a cold cache), so they
                    // are not counted: with them outstanding the wait holds a little longer, never too short.
                    lds::waitCopiesAndReads<(S - 3u) * Cfg::Copies + Cfg::CopiesA>();
                    lds::barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    issueB(slot, adv);
                    readFrags(f0, (i + 1u) % S, 0u);
                    multiplyScaled(f1, std::integral_constant<uint32_t, parity * 2u + 1u>{});
                    scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                    scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::CopiesB>();
                    __builtin_amdgcn_sched_barrier(0);
                };
                for(uint32_t i = 0; i < stages; i += 2u)
                {
                    sA.load(sA.next, i / 2u + 1u < mx.pairs ? i / 2u + 1u : mx.pairs - 1u);
                    sB.load(sB.next, i / 2u + 1u < mx.pairs ? i / 2u + 1u : mx.pairs - 1u);
                    __builtin_amdgcn_sched_barrier(0);
                    stage(i, std::integral_constant<uint32_t, 0u>{});
                    if(i + 1u < stages)
                        stage(i + 1u, std::integral_constant<uint32_t, 1u>{});
                    sA.take(sA.next, i / 2u + 1u);
                    sB.take(sB.next, i / 2u + 1u);
                }
                lds::waitCopiesAndReads<0u>(); // the surplus copies still target this workgroup's LDS
                lds::barrier();
            }
            else if constexpr(Cfg::KSteps == 2u)
            {
                // Prologue
#pragma unroll
                for(uint32_t s = 0; s < S - 1u; ++s)
                    issueStage(s);
                lds::waitCopiesAndReads<(S - 2u) * Cfg::Copies>();
                lds::barrier();
                Frags f0, f1;
                readFrags(f0, 0u, 0u);

                // Steady state: a new stage is issued every iteration
                uint32_t i = 0;
                for(; i + (S - 1u) < stages; ++i)
                {
                    if constexpr(!Cfg::AKMajor || !Cfg::BKMajor)
                    {
                        lds::waitReads(); // fragments read during the previous phase
                        pinFrags(f0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    issueA((i + S - 1u) % S);
                    readFrags(f1, i % S, 1u);
                    multiply(f0);
                    // LDS reads ride on the first half of the MFMAs (so they are back at the
                    // barrier), the copies on the second half, two MFMAs per copy
                    scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                    scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::CopiesA>();
                    __builtin_amdgcn_sched_barrier(0); // nothing moves across the synchronisation point
                    // stage i+1 has landed once only stage i+2 and the A half of stage i+3 are in flight
                    lds::waitCopiesAndReads<(S - 3u) * Cfg::Copies + Cfg::CopiesA>();
                    pinFrags(f1);
                    lds::barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    issueB((i + S - 1u) % S);
                    readFrags(f0, (i + 1u) % S, 0u);
                    multiply(f1);
                    scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();
                    scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::CopiesB>();
                    __builtin_amdgcn_sched_barrier(0);
                }
                // Drain: nothing left to issue; the remaining stages are already in flight
                for(; i < stages; ++i)
                {
                    const bool more = i + 1u < stages;
                    if constexpr(!Cfg::AKMajor || !Cfg::BKMajor)
                    {
                        lds::waitReads();
                        pinFrags(f0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    readFrags(f1, i % S, 1u);
                    multiply(f0);
                    __builtin_amdgcn_sched_barrier(0);
                    lds::waitCopiesAndReads<0u>();
                    pinFrags(f1);
                    lds::barrier();
                    __builtin_amdgcn_sched_barrier(0);
                    if(more)
                        readFrags(f0, (i + 1u) % S, 0u);
                    multiply(f1);
                }
            }
            else
            {
                // One MFMA step per stage (fp8 in 64-byte stages): a phase multiplies stage s (fragments read
                // during the previous phase) while it reads the fragments of stage s+1 and issues
                // the copies of stage s+3; the wait + barrier closing the phase makes stage s+2
                // visible.  Two phases per loop trip so the fragment sets swap without copies.
                // Every phase issues a stage, so the loop body and its wait counts are uniform:
                // past the end of K the last stage is copied again into a ring slot nobody reads.
                static_assert(S == 4u && Cfg::KSteps == 1u, "ring of four, one MFMA step per stage");
                Frags f0, f1;
#define ROCWMMA_AMD_PHASE(STAGE, CUR, NXT)                                                               \
    do                                                                                                  \
    {                                                                                                   \
        issueStage(((STAGE) + S - 1u) % S, (STAGE) + S < stages);                                       \
        readFrags(NXT, ((STAGE) + 1u) % S, 0u);                                                         \
        multiply(CUR);                                                                                  \
        scheduleInterleaved<Cfg::MfmasPerStep / 2u, Cfg::ReadsPerStep, 0u>();                           \
        scheduleInterleaved<Cfg::MfmasPerStep - Cfg::MfmasPerStep / 2u, 0u, Cfg::Copies>();             \
        __builtin_amdgcn_sched_barrier(0);                                                              \
        lds::waitCopiesAndReads<(S - 3u) * Cfg::Copies>();                                              \
        pinFrags(NXT);                                                                                  \
        lds::barrier();                                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                              \
    } while(0)

#pragma unroll
                for(uint32_t s = 0; s < S - 1u; ++s)
                    issueStage(s, s + 1u < stages);
                lds::waitCopiesAndReads<(S - 3u) * Cfg::Copies>(); // stages 0 and 1 have landed
                lds::barrier();
                readFrags(f0, 0u, 0u);
                if constexpr(!Cfg::AKMajor || !Cfg::BKMajor)
                {
                    lds::waitReads(); // the transposing reads are outside the compiler's tracking
                    pinFrags(f0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                uint32_t s = 0;
                for(; s + 1u < stages; s += 2u)
                {
                    ROCWMMA_AMD_PHASE(s, f0, f1);
                    // (past the last stage this reads a ring slot whose content nobody multiplies:
                    // an unconditional phase body keeps the instruction interleave intact)
                    ROCWMMA_AMD_PHASE(s + 1u, f1, f0);
                }
                if(s < stages)
                    multiply(f0);
                lds::waitCopiesAndReads<0u>(); // the surplus copies still target this workgroup's LDS
                lds::barrier();
#undef ROCWMMA_AMD_PHASE
            }

            if constexpr(Part != TilePart::Whole)
            {
                // Part of a tile's K range (stream-K).  A contributor hands its raw accumulators over
                // through its workspace slot and is done; the owner (the part that starts at K = 0)
                // adds the slots of the parts behind it, in order, and goes on to the epilogue.
                if(streamKHandOver<Cfg, Part>(acc, sk))
                    return;
            }

            if constexpr(!std::is_same<Emit, Epilogue>::value)
            {
                emit(acc, row0 + waveM * Cfg::WaveM, col0 + waveN * Cfg::WaveN);
                return;
            }
            else
            {
                (void)emit;
            }
            // Epilogue: D = alpha * acc + beta * C, one row of blocks (BlocksN blocks) at a time,
            // 16-byte accesses per lane.  Every block of a group has registers of its own, so
            // the stores of a group issue back to back (a store whose data registers are about
            // to be overwritten holds up the instruction stream until it has read them), and
            // the C blocks of the next two groups are in flight while a group is finished.
            const uint32_t wRow        = row0 + waveRow;
            const uint32_t wCol        = col0 + waveN * Cfg::WaveN;
            // Plain stores: the 32-byte pieces a store instruction writes per row are merged into
            // full lines in the L2.  Non-temporal stores bypass that merge and were 3-5x slower
            // (4096 x 14336 x 256 int8: 157-277 us against 58 us).
            // (accumulator layout: lane l owns runs of 4 consecutive columns of row l % Block;
            // 32-wide blocks: 4 runs at columns 8 r + 4 (l / 32); 16-wide blocks: 1 run at 4 (l / 16))
            constexpr uint32_t Runs     = Cfg::Block == 32u ? 4u : 1u; // runs per block per lane
            const uint32_t     accRow   = lane & (Cfg::Block - 1u);
            const uint32_t     accGroup = lane / Cfg::Block; // 0..1 or 0..3
            // (edge tiles: a lane's run of four columns of one row is inside the problem or outside it
            // as a whole, N being a multiple of 16)
            auto inside = [&](uint32_t bi, uint32_t bj, uint32_t r) {
                return wRow + blockRow(bi) + accRow < m && wCol + bj * Cfg::Block + 8u * r + 4u * accGroup < n;
            };
            auto storeBlock = [&](uint32_t bi, uint32_t bj, auto const& f) {
                typedef uint32_t Words __attribute__((ext_vector_type(sizeof(OutT))));
                OutT* dst = d + static_cast<size_t>(wRow + blockRow(bi)) * ldd + wCol + bj * Cfg::Block;
#pragma unroll
                for(uint32_t r = 0; r < Runs; ++r)
                {
                    Words v;
                    __builtin_memcpy(&v, f.x + 4u * r, sizeof(v));
                    if(!Cfg::Edges || inside(bi, bj, r))
                        *reinterpret_cast<Words*>(dst + static_cast<size_t>(accRow) * ldd + 8u * r + 4u * accGroup) = v;
                }
            };
            auto loadBlockC = [&](uint32_t bi, uint32_t bj, auto& f) {
                const OutT* src = c + static_cast<size_t>(wRow + blockRow(bi)) * ldc + wCol + bj * Cfg::Block;
                if constexpr(!Cfg::Edges)
                    load_matrix_sync(f, src, ldc);
                else
                {
                    typedef uint32_t Words __attribute__((ext_vector_type(sizeof(OutT))));
#pragma unroll
                    for(uint32_t r = 0; r < Runs; ++r)
                    {
                        Words v = {};
                        if(inside(bi, bj, r))
                            v = *reinterpret_cast<const Words*>(src + static_cast<size_t>(accRow) * ldc + 8u * r + 4u * accGroup);
                        __builtin_memcpy(f.x + 4u * r, &v, sizeof(v));
                    }
                }
            };
            // 16-bit outputs with 16-wide blocks: a lane's run is only 8 bytes, a store instruction would
            // write 32-byte pieces.  Two neighbouring blocks are handled together: v_permlane16_swap
            // exchanges the second block's run of a lane in an even 16-lane row with the first block's
            // run of its partner in the next row, after which every lane owns 8 consecutive columns
            // (even rows: of the first block, odd rows: of the second) and moves 16 bytes; an
            // instruction then covers 64 contiguous bytes per matrix row.  The exchange is its own
            // inverse, so C is read the same way.
            constexpr bool PairIO = Cfg::Block == 16u && sizeof(OutT) == 2u && Cfg::BlocksN % 2u == 0u;
            const uint32_t pairCol = (accGroup & 1u) * 16u + 4u * (accGroup & 2u);
            auto           blockOffset = [&](uint32_t bi, uint32_t bj, uint32_t ld) {
                return static_cast<size_t>(wRow + blockRow(bi)) * ld + wCol + bj * Cfg::Block;
            };
            auto swapPair = [](auto& fx, auto& fy) {
                uint32_t x[2], y[2];
                __builtin_memcpy(x, fx.x, 8);
                __builtin_memcpy(y, fy.x, 8);
#pragma unroll
                for(uint32_t w = 0; w < 2u; ++w)
                {
                    auto r = __builtin_amdgcn_permlane16_swap(x[w], y[w], false, false);
                    x[w]   = r[0];
                    y[w]   = r[1];
                }
                __builtin_memcpy(fx.x, x, 8);
                __builtin_memcpy(fy.x, y, 8);
            };
            // (edge tiles: a lane's eight columns of one row are inside the problem or outside it as a whole)
            auto insidePair = [&](uint32_t bi, uint32_t bj) {
                return !Cfg::Edges || (wRow + blockRow(bi) + accRow < m && wCol + bj * Cfg::Block + pairCol < n);
            };
            auto storePair = [&](uint32_t bi, uint32_t bj, auto& fx, auto& fy) {
                swapPair(fx, fy);
                typedef uint32_t Words __attribute__((ext_vector_type(4)));
                Words            v;
                __builtin_memcpy(&v, fx.x, 8);
                __builtin_memcpy(reinterpret_cast<char*>(&v) + 8, fy.x, 8);
                if(insidePair(bi, bj))
                    *reinterpret_cast<Words*>(d + blockOffset(bi, bj, ldd) + static_cast<size_t>(accRow) * ldd + pairCol) = v;
            };
            auto loadPair = [&](uint32_t bi, uint32_t bj, auto& fx, auto& fy) {
                typedef uint32_t Words __attribute__((ext_vector_type(4)));
                Words            v = {};
                if(insidePair(bi, bj))
                    v = *reinterpret_cast<const Words*>(c + blockOffset(bi, bj, ldc) + static_cast<size_t>(accRow) * ldc + pairCol);
                __builtin_memcpy(fx.x, &v, 8);
                __builtin_memcpy(fy.x, reinterpret_cast<const char*>(&v) + 8, 8);
                swapPair(fx, fy);
            };
            // Fused configurations: the bias values of a lane's columns of one block are fetched (four
            // consecutive floats per run, cache hits after the first row of blocks) just before the
            // block's results go out.
            static_assert(!Cfg::Fused || std::is_same<CompT, float>::value, "fused epilogue: f32 compute");
            struct BiasOfBlock
            {
                float v[Cfg::Fused ? 4u * Runs : 1u];
            };
            auto loadBias = [&](uint32_t bj) {
                BiasOfBlock bv = {};
                if constexpr(Cfg::Fused)
                {
                    if(ex.fused.bias)
                    {
#pragma unroll
                        for(uint32_t r = 0; r < Runs; ++r)
                        {
                            const uint32_t col = wCol + bj * Cfg::Block + 8u * r + 4u * accGroup;
                            if(!Cfg::Edges || col < n)
                                __builtin_memcpy(&bv.v[4u * r], ex.fused.bias + col, 16);
                        }
                    }
                }
                return bv;
            };
            // With 16-wide blocks a wave's bias values (four per block and lane) are few enough to be fetched once,
            // in front of everything else the epilogue requests, and kept for every row of blocks; fetched per
            // block, each load's latency sat in front of that block's stores (8192^3 f16 with a bias: +26 us,
            // hoisted: +3 us).  The 32-wide blocks (16 values per block and lane) keep the per-block loads: held
            // for all blocks they spilled.
            constexpr bool HoistBias = Cfg::Fused && 4u * Runs * Cfg::BlocksN <= 32u;
            BiasOfBlock    biasRow[HoistBias ? Cfg::BlocksN : 1u];
            if constexpr(HoistBias)
            {
#pragma unroll
                for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                    biasRow[bj] = loadBias(bj);
                __builtin_amdgcn_sched_barrier(0);
            }
            auto biasOf = [&](uint32_t bj) {
                if constexpr(HoistBias)
                    return biasRow[bj];
                else
                    return loadBias(bj);
            };
            // What the results of `Count` blocks of a row from block `first` on pass through: at once, but for 32-wide blocks (16 values
            // per block and lane), which spilled.  Those keep a branch on the activation per value where there is a C: e4m3 with bias,
            // a branch per value and one per block, us: 1280 x 4608 x 256 A col / B row 15.0, 17.3; 912 x 6432 x 256 14.6, 16.4; with GELU 16.8, 15.3;
            // 1024 x 7040 x 768 both row-major 21.1, 22.0, with GELU 21.6, 24.2.  Without C one branch is the faster one: 11.9, 11.5; 12.1, 11.4;
            // 16.7, 15.7.
            auto finish = [&](uint32_t bi, uint32_t first, auto countC, auto withC) {
                if constexpr(Cfg::Fused)
                {
                    constexpr uint32_t Count = decltype(countC)::value, Per = Cfg::FragAcc::num_elements;
                    constexpr uint32_t Group = Cfg::Block == 16u ? Count : 1u;
#pragma unroll
                    for(uint32_t from = 0; from < Count; from += Group)
                    {
                        float v[Group * Per];
#pragma unroll
                        for(uint32_t j = 0; j < Group; ++j)
                        {
                            const BiasOfBlock bv = biasOf(first + from + j);
#pragma unroll
                            for(uint32_t e = 0; e < Per; ++e)
                                v[j * Per + e] = acc[bi][first + from + j].x[e] + bv.v[e];
                        }
                        if constexpr(Cfg::Block == 32u && decltype(withC)::value)
                        {
#pragma unroll
                            for(uint32_t i = 0; i < Group * Per; ++i)
                            {
                                float one[1] = {v[i]};
                                applyActivation(one, ex.fused.activation);
                                v[i] = one[0];
                            }
                        }
                        else
                            applyActivation(v, ex.fused.activation);
#pragma unroll
                        for(uint32_t j = 0; j < Group; ++j)
#pragma unroll
                            for(uint32_t e = 0; e < Per; ++e)
                                acc[bi][first + from + j].x[e] = v[j * Per + e];
                    }
                }
                (void)bi, (void)first, (void)countC, (void)withC;
            };
            constexpr std::true_type  withC{};
            constexpr std::false_type withoutC{};
            constexpr std::integral_constant<uint32_t, Cfg::BlocksN> wholeRow{};
            if(beta != static_cast<CompT>(0))
            {
                if constexpr(Cfg::StagedC)
                {
                    // C reaches the accumulator layout through LDS: whole-wave direct copies
                    // fetch full rows of a 32-row group of GroupBlocks blocks (read in the
                    // accumulator layout straight from global memory, an instruction would touch
                    // 32 rows for 32 bytes each, at half the rate).  Row r is stored with its
                    // 16-byte chunks XOR-swizzled by r % 16 so that the 16 rows a quarter-wave
                    // reads at one chunk position fall into distinct bank groups.  The main-loop
                    // ring is free by now and every wave owns two group buffers in it.
                    constexpr uint32_t GB          = Cfg::GroupBlocks;
                    constexpr uint32_t RowBytes    = GB * Cfg::Block * sizeof(OutT); // 256 or 512
                    constexpr uint32_t GroupBytes  = Cfg::Block * RowBytes;
                    constexpr uint32_t RowChunks   = RowBytes / 16u;
                    constexpr uint32_t RowsPerCopy = 1024u / RowBytes;
                    constexpr uint32_t CopiesC     = GroupBytes / 1024u;
                    constexpr uint32_t GroupsPerRow = Cfg::BlocksN / GB;
                    constexpr uint32_t NG          = Cfg::BlocksM * GroupsPerRow;
                    constexpr uint32_t Buffers     = Cfg::BuffersC;
                    static_assert((RowBytes == 256u || RowBytes == 512u) && Buffers * GroupBytes * Cfg::Waves <= Cfg::LdsBytes
                                      && NG >= Buffers,
                                  "C staging geometry");
                    char*          myLds  = ldsRaw + wave * (Buffers * GroupBytes);
                    const char*    cWave  = reinterpret_cast<const char*>(c + static_cast<size_t>(wRow) * ldc + wCol);
                    const size_t   ldcB   = static_cast<size_t>(ldc) * sizeof(OutT);
                    const uint32_t cpRow  = lane / RowChunks; // row inside a copy
                    const uint32_t chunk  = lane % RowChunks; // chunk position inside the LDS row
                    auto           copyGroup = [&](uint32_t gi) {
                        const uint32_t bi = gi / GroupsPerRow, bj0 = (gi % GroupsPerRow) * GB;
#pragma unroll
                        for(uint32_t i = 0; i < CopiesC; ++i)
                        {
                            const uint32_t r = RowsPerCopy * i + cpRow;
                            const char*    src;
                            if constexpr(Cfg::RolledRows) // (what does not depend on bi stays in front of the loop)
                                src = cWave + blockRow(bi) * ldcB + (r * ldcB + ((chunk ^ (r & 15u)) << 4));
                            else if constexpr(!Cfg::Edges)
                                src = cWave + (blockRow(bi) + r) * ldcB + bj0 * Cfg::Block * sizeof(OutT) + ((chunk ^ (r & 15u)) << 4);
                            else
                            {
                                // (rows and columns past the problem's fetch some element of C, used by nobody)
                                const uint32_t row  = wRow + blockRow(bi) + r;
                                const uint32_t colB = (wCol + bj0 * Cfg::Block) * static_cast<uint32_t>(sizeof(OutT)) + ((chunk ^ (r & 15u)) << 4);
                                src = reinterpret_cast<const char*>(c) + static_cast<size_t>(row < m ? row : m - 1u) * ldcB
                                      + (colB < n * static_cast<uint32_t>(sizeof(OutT)) ? colB : 0u);
                            }
                            lds::asyncCopy16Streaming(myLds + (gi % Buffers) * GroupBytes + i * 1024u, src);
                        }
                    };
                    const uint32_t rdRow  = accRow;
                    const uint32_t rdBase = rdRow * RowBytes;
#pragma unroll
                    for(uint32_t gi = 0; gi < Buffers; ++gi)
                        copyGroup(gi);
                    static_assert(!Cfg::RolledRows || (GroupsPerRow == 1u && !Cfg::Edges), "a row of blocks is one group of C");
#pragma unroll Cfg::RolledRows ? 1u : NG
                    for(uint32_t gi = 0; gi < NG; ++gi)
                    {
                        const uint32_t bi = gi / GroupsPerRow, bj0 = (gi % GroupsPerRow) * GB, at = Cfg::RolledRows ? 0u : bi;
                        // (the stores of D do not count, see copy_waits.hpp)
                        const uint32_t inFlight = stagedCInFlight(gi, NG, CopiesC, Buffers); // (a constant where the loop is unrolled)
                        constexpr uint32_t Three = Buffers == 4u ? 3u * CopiesC : 0u, Two = Buffers == 4u ? 2u * CopiesC : 0u;
                        if(Buffers == 4u && inFlight == Three)
                            lds::waitCopiesAndReads<Three>();
                        else if(Buffers == 4u && inFlight == Two)
                            lds::waitCopiesAndReads<Two>();
                        else if(inFlight != 0u)
                            lds::waitCopiesAndReads<CopiesC>();
                        else
                            lds::waitCopiesAndReads<0u>();
                        asm volatile("" ::: "memory");
                        if(!Cfg::RolledRows && gi % GroupsPerRow == 0u)
                            takeRow(bi, at);
                        typename Cfg::FragC io[GB];
#pragma unroll
                        for(uint32_t bj = 0; bj < GB; ++bj)
#pragma unroll
                            for(uint32_t r = 0; r < Runs; ++r)
                            {
                                // logical chunk of this run: block bj holds Block / 4 chunks per row
                                const uint32_t g = bj * (Cfg::Block / 4u) + 2u * r + accGroup;
                                detail::copyBytes<16u>(io[bj].x + 4u * r,
                                                       myLds + (gi % Buffers) * GroupBytes + rdBase + ((g ^ (rdRow & 15u)) << 4));
                            }
                        if constexpr(Cfg::RolledRows)
                            takeRow(bi, at); // (behind the reads: its branches pass while they are under way)
#pragma unroll
                        for(uint32_t bj = 0; bj < GB; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < io[bj].num_elements; ++e)
                                acc[at][bj0 + bj].x[e] = alpha * acc[at][bj0 + bj].x[e] + beta * static_cast<CompT>(io[bj].x[e]);
                        finish(at, bj0, std::integral_constant<uint32_t, GB>{}, withC);
                        // (results replace the accumulators: every store has registers of its own)
#pragma unroll
                        for(uint32_t bj = 0; bj < GB; ++bj)
                            storeBlock(bi, bj0 + bj, acc[at][bj0 + bj]);
                        __builtin_amdgcn_sched_barrier(0);
                        // behind the stores: the next wait then leaves these copies in flight and not the stores
                        if(gi + Buffers < NG)
                        {
                            lds::waitReads(); // the buffer is overwritten next
                            asm volatile("" ::: "memory");
                            copyGroup(gi + Buffers);
                        }
                    }
                }
                else if constexpr(Cfg::PrefetchC)
                {
#pragma unroll
                    for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                    {
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < early[bi][bj].num_elements; ++e)
                                acc[bi][bj].x[e] = alpha * acc[bi][bj].x[e] + beta * static_cast<CompT>(early[bi][bj].x[e]);
                        finish(bi, 0u, wholeRow, withC);
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                        {
                            auto& io = early[bi][bj];
#pragma unroll
                            for(uint32_t e = 0; e < io.num_elements; ++e)
                                io.x[e] = narrowed<OutT>(acc[bi][bj].x[e]);
                            if constexpr(!PairIO)
                                storeBlock(bi, bj, io);
                            else if(bj % 2u == 1u)
                                storePair(bi, bj - 1u, early[bi][bj - 1u], io);
                        }
                    }
                }
                else if constexpr(Cfg::WideWave)
                {
                    // 16- and 8-bit C: all of the wave's C is requested at once, 16 to 64 loads that the only wave of its SIMD has in flight (two rows
                    // of blocks ahead, as below, was half as much per compute unit as with eight waves).  Edge tiles: rows and columns past the
                    // problem's fetch some element of C, used by nobody; a branch around every load cost more than the loads.  1040 x 6000 x 256, C
                    // and D f16: eight waves of 64 x 64 11.8 us, two rows ahead 14.8, at once 10.9; C and D int8, K = 512, 14.9, 19.1, 13.2; on whole
                    // tiles, 4096^3 f16, 110.6, 102.8, 101.6.
                    constexpr uint32_t Pieces = PairIO ? Cfg::BlocksN / 2u : Cfg::BlocksN; // of a row of blocks
                    typedef uint32_t   Words __attribute__((ext_vector_type(PairIO ? 4u : sizeof(OutT))));
                    // (with the fused epilogue at most 64 registers of it, the rows behind them as soon as theirs are free: all of them spill)
                    constexpr uint32_t PerRow = Pieces * sizeof(Words) / 4u, Ahead = Cfg::Fused && PerRow > 8u ? Cfg::BlocksM / 2u : Cfg::BlocksM;
                    Words              raw[Ahead][Pieces];
                    auto               loadRow = [&](uint32_t bi) {
                        const uint32_t row = wRow + blockRow(bi) + accRow;
                        const OutT*    src = c + static_cast<size_t>(Cfg::Edges && row >= m ? m - 1u : row) * ldc;
#pragma unroll
                        for(uint32_t p = 0; p < Pieces; ++p)
                        {
                            const uint32_t col = wCol + (PairIO ? 2u * p * Cfg::Block + pairCol : p * Cfg::Block + 4u * accGroup);
                            raw[bi % Ahead][p] = *reinterpret_cast<const Words*>(src + (Cfg::Edges && col >= n ? 0u : col));
                        }
                    };
#pragma unroll
                    for(uint32_t bi = 0; bi < Ahead; ++bi)
                        loadRow(bi);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                    {
                        takeRow(bi, bi);
                        Words row[Pieces];
#pragma unroll
                        for(uint32_t p = 0; p < Pieces; ++p)
                            row[p] = raw[bi % Ahead][p];
                        if(bi + Ahead < Cfg::BlocksM)
                            loadRow(bi + Ahead);
                        typename Cfg::FragC io[Cfg::BlocksN];
#pragma unroll
                        for(uint32_t p = 0; p < Pieces; ++p)
                        {
                            if constexpr(PairIO)
                            {
                                __builtin_memcpy(io[2u * p].x, &row[p], 8);
                                __builtin_memcpy(io[2u * p + 1u].x, reinterpret_cast<const char*>(&row[p]) + 8, 8);
                                swapPair(io[2u * p], io[2u * p + 1u]);
                            }
                            else
                                __builtin_memcpy(io[p].x, &row[p], sizeof(Words));
                        }
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < Cfg::FragC::num_elements; ++e)
                                acc[bi][bj].x[e] = alpha * acc[bi][bj].x[e] + beta * static_cast<CompT>(io[bj].x[e]);
                        finish(bi, 0u, wholeRow, withC);
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < Cfg::FragC::num_elements; ++e)
                                io[bj].x[e] = narrowed<OutT>(acc[bi][bj].x[e]);
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                        {
                            if constexpr(!PairIO)
                                storeBlock(bi, bj, io[bj]);
                            else if(bj % 2u == 1u)
                                storePair(bi, bj - 1u, io[bj - 1u], io[bj]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                else
                {
                typename Cfg::FragC fc[2][Cfg::BlocksN];
                auto                loadGroup = [&](uint32_t bi) {
                    if constexpr(PairIO)
                    {
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; bj += 2u)
                            loadPair(bi, bj, fc[bi % 2u][bj], fc[bi % 2u][bj + 1u]);
                    }
                    else
                    {
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                            loadBlockC(bi, bj, fc[bi % 2u][bj]);
                    }
                };
                loadGroup(0u);
                if constexpr(Cfg::BlocksM > 1u)
                    loadGroup(1u);
#pragma unroll
                for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                {
#pragma unroll
                    for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                        for(uint32_t e = 0; e < Cfg::FragC::num_elements; ++e)
                            acc[bi][bj].x[e] = alpha * acc[bi][bj].x[e] + beta * static_cast<CompT>(fc[bi % 2u][bj].x[e]);
                    finish(bi, 0u, wholeRow, withC);
#pragma unroll
                    for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                        for(uint32_t e = 0; e < Cfg::FragC::num_elements; ++e)
                            fc[bi % 2u][bj].x[e] = narrowed<OutT>(acc[bi][bj].x[e]);
                    if constexpr(PairIO)
                    {
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; bj += 2u)
                            storePair(bi, bj, fc[bi % 2u][bj], fc[bi % 2u][bj + 1u]);
                    }
                    else
                    {
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                            storeBlock(bi, bj, fc[bi % 2u][bj]);
                    }
                    if(bi + 2u < Cfg::BlocksM)
                        loadGroup(bi + 2u);
                    __builtin_amdgcn_sched_barrier(0);
                }
                }
            }
            else
            {
#pragma unroll Cfg::RolledRows ? 1u : Cfg::BlocksM
                for(uint32_t bi = 0; bi < Cfg::BlocksM; ++bi)
                {
                    const uint32_t at = Cfg::RolledRows ? 0u : bi;
                    takeRow(bi, at);
                    if constexpr(std::is_same<OutT, CompT>::value)
                    {
                        // results replace the accumulators, so no two stores share data registers
                        // (with alpha = 1 they go out as they are: a 32-bit integer multiply runs at a quarter of the
                        // rate of the other vector instructions, 128 of them per lane and tile)
                        if(Cfg::Fused || alpha != static_cast<CompT>(1))
                        {
#pragma unroll
                            for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                                for(uint32_t e = 0; e < acc[at][bj].num_elements; ++e)
                                    acc[at][bj].x[e] = alpha * acc[at][bj].x[e];
                            finish(at, 0u, wholeRow, withoutC);
                        }
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                            storeBlock(bi, bj, acc[at][bj]);
                    }
                    else
                    {
                        typename Cfg::FragC fd[Cfg::BlocksN];
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < fd[bj].num_elements; ++e)
                                acc[at][bj].x[e] = alpha * acc[at][bj].x[e];
                        finish(at, 0u, wholeRow, withoutC);
#pragma unroll
                        for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
#pragma unroll
                            for(uint32_t e = 0; e < fd[bj].num_elements; ++e)
                                fd[bj].x[e] = narrowed<OutT>(acc[at][bj].x[e]);
                        if constexpr(PairIO)
                        {
#pragma unroll
                            for(uint32_t bj = 0; bj < Cfg::BlocksN; bj += 2u)
                                storePair(bi, bj, fd[bj], fd[bj + 1u]);
                        }
                        else
                        {
#pragma unroll
                            for(uint32_t bj = 0; bj < Cfg::BlocksN; ++bj)
                                storeBlock(bi, bj, fd[bj]);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }

    } // namespace
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_BLOCKED_CORE_HPP
