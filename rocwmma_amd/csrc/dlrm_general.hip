// DLRM dot interaction for the shapes the kernels that hold samples in LDS (dlrm.hip, dlrm_sample.hip) do not take:
// samples larger than the LDS or of more than 192 feature rows.  The reference's tests run
// (m, k) = (1024, 1024) among others (test/dlrm/test/dlrm_test_params.hpp:51-68); semantics = dlrm_fwd_CPU /
// dlrm_bwd_CPU (test/reference_impl.hpp:83-179).
//
// A sample of that size is a matrix product of its own (1024 x 1024 x 1024), so a sample's work is cut into tiles
// of 128 x 128 over workgroups of four waves (2 x 2, 64 x 64 each, 32 x 32 blocks), one grid for the whole batch:
//
//   * forward: tile (I, J), J <= I, of Z = F F^T; both operands are rows of F with K contiguous.  The strict lower
//     triangle leaves through a 32 x 32 LDS block per wave as row pieces, which are contiguous in the packed
//     output.  No m x m scratch in global memory.  (float32, and float16 where 128 feature rows span 2 GiB; other float16
//     samples: dlrm_general_fwd.hip.)
//   * backward: tile (I, N) of grad = S F, S = the symmetric matrix with zero diagonal whose strict lower triangle
//     is the packed upstream gradient, never materialised: where the contraction index lies below the tile's rows
//     the packed triangle holds S row by row, where it lies above them it holds the transpose, and only the
//     stages that meet the diagonal are gathered element by element (float32; float16 has a kernel of its own that
//     takes them out of the packed triangle as they lie, with tiles of up to 256 x 256).
//
// Operands go through LDS (coalesced 16-byte pieces into registers one stage ahead, then LDS, then fragments).
// Rows from m on and columns from k on are never read: their lanes multiply zeros.
#include "common.hpp"
#include <utility>
#include <rocwmma/rocwmma_lds.hpp>
#include <rocwmma/rocwmma_transforms.hpp>

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchDlrmFwdTilesF16(const void* input, void* output, uint32_t m, uint32_t k, uint32_t batch, hipStream_t stream);

    namespace
    {
        typedef uint32_t u32x4_t __attribute__((ext_vector_type(4), may_alias));
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2), may_alias));
        typedef float    f32x4_t __attribute__((ext_vector_type(4), may_alias));

        constexpr uint32_t kTile       = 128; // workgroup tile edge
        constexpr uint32_t kWaveTile   = 64;
        constexpr uint32_t kMaxRows    = 32768; // m * (m - 1) stays below 2^32
        constexpr uint32_t kNowhere    = 0x80000000u; // beyond every sample: a bounds-checked load there returns zero

        // offset of Z(row, 0) in a sample's packed output / upstream row
        ROCWMMA_DEVICE inline size_t packedRow(uint32_t k, uint32_t row)
        {
            return static_cast<size_t>(k) + (static_cast<size_t>(row) * (row - (row != 0u))) / 2u;
        }

        ROCWMMA_DEVICE inline void waveSync()
        {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }

        // Which (sample, tile) a workgroup takes.  Workgroups are handed to the device's 8 XCDs in turn (workgroup w
        // runs on XCD w % 8), and every XCD has an L2 of its own: all tiles of a sample go to one XCD, sample s to XCD
        // s % 8, so that a sample's operands are fetched into one L2 once instead of into all eight (measured at
        // (1024, 1024, 64) in f16: 955 MiB fetched per forward launch for 128 MiB of features with the tiles of a
        // sample dealt out over the XCDs).  The grid is 8 * ceil(batch / 8) * tiles workgroups.
        constexpr uint32_t kXcds = 8;
        ROCWMMA_DEVICE inline void sampleAndTile(uint32_t tiles, uint32_t& sample, uint32_t& tile)
        {
            const uint32_t slot = blockIdx.x / kXcds;
            sample              = (slot / tiles) * kXcds + blockIdx.x % kXcds;
            tile                = slot % tiles;
        }

        // ------------------------------------------------------------------ operands through LDS
        // In the fragment layout consecutive lanes hold different rows, and a global load whose lanes touch 32
        // different cache lines is served at a fraction of the rate of one whose lanes read consecutive addresses
        // (with operands straight from global memory the f16 forward kernel ran at half the rate at (1024, 1024, 64)).  So a thread fetches consecutive 16-byte pieces of a tile row into registers (one
        // stage ahead of the multiplication), the pieces go to LDS, and the fragments come from there.
        //
        // "rows" layout: 128 tile rows of 128 bytes of K (row pitch 144 bytes: 16-byte aligned, rows spread over the banks);
        // a fragment is one 16-byte read per lane.  Both operands of the forward kernel, S of the float32 backward kernel
        // where the packed triangle holds it row by row (contraction index below the tile's rows).
        constexpr uint32_t kRowPitch  = 144;
        constexpr uint32_t kRowsBytes = kTile * kRowPitch; // 18432

        // 16 bytes at a 2-byte aligned address (rows of the packed triangle start anywhere)
        struct __attribute__((packed, aligned(2))) UnalignedPiece
        {
            uint32_t w[4];
        };
        ROCWMMA_DEVICE inline u32x4_t loadUnaligned(const float16_t* from)
        {
            const UnalignedPiece p = *reinterpret_cast<const UnalignedPiece*>(from);
            return u32x4_t{p.w[0], p.w[1], p.w[2], p.w[3]};
        }

        using FragK16   = fragment<matrix_a, 32, 32, 16, float16_t, row_major>;
        using FragAcc16 = fragment<accumulator, 32, 32, 16, float32_t>;

        // fragment words of 32-row block `block32` (of the tile's 128 rows) at K step `ks` (16 halves) of a "rows" tile
        ROCWMMA_DEVICE inline u32x4_t rowsFragment(const char* tile, uint32_t block32, uint32_t ks, uint32_t lane)
        {
            return *reinterpret_cast<const u32x4_t*>(tile + (block32 * 32u + (lane & 31u)) * kRowPitch + ks * 32u + (lane >> 5) * 16u);
        }

        // the fragment instruction `w` of a 16-byte piece takes: all of it (eight halves) or its word w (one float)
        template <typename Frag>
        ROCWMMA_DEVICE inline Frag pieceFragment(const u32x4_t& piece, uint32_t w)
        {
            Frag f;
            if constexpr(Frag::num_elements == 8u)
                *reinterpret_cast<u32x4_t*>(f.x) = piece;
            else
            {
                // (through a named scalar: __builtin_bit_cast applied to the element expression itself reads element 0)
                const uint32_t word = piece[w];
                f.x[0]              = __builtin_bit_cast(float, word);
            }
            return f;
        }

        // T = float16_t: 64 of K per stage, one v_mfma_f32_32x32x16_f16 per 16-byte piece and block; T = float: 32 of K
        // per stage, four v_mfma_f32_32x32x2_f32 per piece and block, one per word (the order in which K is contracted
        // is free as long as both multiplicands agree: instruction t of a piece contracts word t of both lane halves)
        template <typename T>
        __global__ void __launch_bounds__(256, sizeof(T) == 2u ? 4 : 3) // (waves per SIMD that fit without spills)
            dlrmFwdStagedKernel(const T* __restrict__ input, T* __restrict__ output, uint32_t m, uint32_t k, uint32_t batch, uint32_t tiles)
        {
            constexpr uint32_t KI = sizeof(T) == 2u ? 16u : 2u;
            using FragK           = fragment<matrix_a, 32, 32, KI, T, row_major>;
            using FragAcc         = fragment<accumulator, 32, 32, KI, float32_t>;
            using AccMap          = detail::AccMap<32, 32, 32>;
            constexpr uint32_t Size     = static_cast<uint32_t>(sizeof(T));
            constexpr uint32_t PerPiece = 16u / Size; // elements of a 16-byte piece
            constexpr uint32_t StageK   = 128u / Size; // a tile row of a stage is 128 bytes
            constexpr uint32_t InstrPerPiece = PerPiece / FragK::num_elements; // 1 or 4
            __shared__ __attribute__((aligned(16))) char lds[2u * kRowsBytes];
            char* const ldsA = lds;
            char* const ldsB = lds + kRowsBytes;

            uint32_t sample, t; // t: tiles of the lower triangle, row by row
            sampleAndTile(tiles, sample, t);
            if(sample >= batch) // (the whole workgroup)
                return;
            const uint32_t tid  = threadIdx.x;
            const uint32_t lane = tid & 63u;
            const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

            uint32_t       I = static_cast<uint32_t>((__builtin_sqrtf(8.0f * static_cast<float>(t) + 1.0f) - 1.0f) * 0.5f);
            while(I * (I + 1u) / 2u > t)
                --I;
            while((I + 1u) * (I + 2u) / 2u <= t)
                ++I;
            const uint32_t J  = t - I * (I + 1u) / 2u;
            const uint32_t I0 = I * kTile, J0 = J * kTile;

            const size_t     width = packedRow(k, m);
            const T* feat = input + static_cast<size_t>(sample) * m * k;
            T*       out  = output + static_cast<size_t>(sample) * width;

            if(t == 0u) // bottom-MLP row: the sample's first feature row
                for(uint32_t e = tid; e < k; e += 256u)
                    out[e] = feat[e];

            const uint32_t wr = wave >> 1, wc = wave & 1u;
            const uint32_t R0 = I0 + wr * kWaveTile, C0 = J0 + wc * kWaveTile;
            // the wave's 64 x 64 holds entries below the diagonal and inside the matrix (every wave stages and meets
            // the barriers all the same)
            const bool waveLive = R0 < m && C0 < min(R0 + kWaveTile - 1u, m - 1u);

            // this thread's pieces of a stage: tile rows tid / 8 + 32 i, piece tid % 8 of the row's 128 bytes.  A row
            // from m on starts at the end of the sample, where a bounds-checked load returns zero.
            const lds::BufferRsrc rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(feat), 0, static_cast<int>(m * k * Size), 0x00020000);
            const uint32_t        pos  = tid & 7u;
            uint32_t              offA[4], offB[4], offLds[4];
#pragma unroll
            for(uint32_t i = 0; i < 4u; ++i)
            {
                const uint32_t r = (tid >> 3) + 32u * i;
                offA[i]          = (min(I0 + r, m) * k + pos * PerPiece) * Size;
                offB[i]          = (min(J0 + r, m) * k + pos * PerPiece) * Size;
                offLds[i]        = r * kRowPitch + pos * 16u;
            }
            u32x4_t ra[4], rb[4];
            auto    fetch = [&](uint32_t k0) {
                const bool inK = k0 + pos * PerPiece < k;
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                {
                    ra[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(inK ? offA[i] + k0 * Size : kNowhere), 0, 0);
                    rb[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(inK ? offB[i] + k0 * Size : kNowhere), 0, 0);
                }
            };

            FragAcc acc[2][2];
#pragma unroll
            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                for(uint32_t j = 0; j < 2u; ++j)
                    fill_fragment(acc[i][j], 0.0f);

            fetch(0u);
#pragma unroll 1
            for(uint32_t k0 = 0; k0 < k; k0 += StageK)
            {
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                {
                    *reinterpret_cast<u32x4_t*>(ldsA + offLds[i]) = ra[i];
                    *reinterpret_cast<u32x4_t*>(ldsB + offLds[i]) = rb[i];
                }
                __syncthreads();
                // the next stage's pieces fly while this one is multiplied (a stage from k on loads nothing)
                fetch(k0 + StageK);
                __builtin_amdgcn_sched_barrier(0);
                if(waveLive)
                {
#pragma unroll
                    for(uint32_t ks = 0; ks < 4u; ++ks) // a row's 128 bytes: 32 per step, 16 per lane half
                    {
                        u32x4_t pa[2], pb[2];
#pragma unroll
                        for(uint32_t i = 0; i < 2u; ++i)
                        {
                            pa[i] = rowsFragment(ldsA, wr * 2u + i, ks, lane);
                            pb[i] = rowsFragment(ldsB, wc * 2u + i, ks, lane);
                        }
#pragma unroll
                        for(uint32_t w = 0; w < InstrPerPiece; ++w)
                        {
                            FragK a[2], b[2];
#pragma unroll
                            for(uint32_t i = 0; i < 2u; ++i)
                            {
                                a[i] = pieceFragment<FragK>(pa[i], w);
                                b[i] = pieceFragment<FragK>(pb[i], w);
                            }
#pragma unroll
                            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                                for(uint32_t j = 0; j < 2u; ++j)
                                    mma_sync(acc[i][j], a[i], applyTranspose(b[j]), acc[i][j]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
            }

            if(!waveLive)
                return;
            // strict lower triangle: block by block through LDS (the operand tiles are done with), then pieces of rows,
            // which are contiguous in the packed output
            T(*st)[33] = reinterpret_cast<T(*)[33]>(lds + wave * (32u * 33u * Size));
            const uint32_t row = lane & 31u, half = lane >> 5;
#pragma unroll
            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                for(uint32_t j = 0; j < 2u; ++j)
                {
                    if(C0 + j * 32u >= min(R0 + i * 32u + 31u, m - 1u)) // (wave uniform: nothing of the block is below the diagonal)
                        continue;
#pragma unroll
                    for(uint32_t e = 0; e < 16u; ++e)
                        st[AccMap::rowOf(e, lane)][AccMap::colOf(e, lane)] = static_cast<T>(acc[i][j].x[e]);
                    waveSync();
#pragma unroll 4
                    for(uint32_t rr = 0; rr < 16u; ++rr)
                    {
                        const uint32_t r = rr * 2u + half, Rg = R0 + i * 32u + r, Cg = C0 + j * 32u + row;
                        if(Rg < m && Cg < Rg)
                            out[packedRow(k, Rg) + Cg] = st[r][row];
                    }
                    waveSync();
                }
        }

        // ------------------------------------------------------------------ float16 backward
        // A workgroup tile of (WavesM * 64) x (BlocksN * 64): WavesM x 2 waves of 64 x (BlocksN * 32), 32 x 32 blocks, 64
        // contraction indices per stage.
        //
        // S is taken in blocks of 64 x 64 that lie below the diagonal, above it or across it: 64 rows of the packed
        // triangle from max(rows, stage) on, 128 contiguous bytes each from column min(rows, stage) on, whichever of the
        // two is the contraction.  Such a block goes to LDS as it is (16-byte pieces through registers: its rows start at
        // any half) and is read back row by row below the diagonal and through the transposing reads above it.  Across
        // the diagonal the entries on and above it are cleared on the way to LDS, and a fragment is the one reading OR-ed
        // with the other.  A wave's 64 rows have one kind per stage, the same two waves carry the block and no other
        // wave's rows need it, so all of this is decided wave by wave.
        //
        // F (contraction index by column) is copied straight into LDS, three stages deep; S has two.  One barrier per
        // stage, in front of its last step: there stage i has been read completely and stage i + 1 has landed, and behind
        // it go out the copies of F(i + 3), the pieces of S(i + 2) into LDS and the loads of S(i + 3).
        //
        // (1024, 1024, 64): 300 -> 185 us (740 TFLOP/s), against 128 x 128 tiles of four waves on one LDS stage with two
        // barriers, gathered element by element across the diagonal.  A stage takes 2.0 us of a compute unit (1070
        // TFLOP/s); the rest is the first loads and the results of a round of tiles, which nothing overlaps.  The matrix
        // pipes are busy 38 % of the time, a wave waits 31 % of it at its LDS reads and barriers; S costs a quarter (148 us with its loads
        // replaced by one address), but neither its alignment (200 us either way) nor its latency: loaded two
        // stages ahead (212), or at a raised wave priority around the matrix instructions (201), it was no faster.
        template <uint32_t WavesM_, uint32_t BlocksN_>
        struct BwdTile
        {
            static constexpr uint32_t WavesM = WavesM_, BlocksN = BlocksN_;
            static constexpr uint32_t Rows = WavesM * 64u, Cols = BlocksN * 64u;
            static constexpr uint32_t Waves = WavesM * 2u, Threads = Waves * 64u;
            static constexpr uint32_t Steps   = 4u; // of 16 contraction indices per stage
            static constexpr uint32_t RingS   = 2u, RingF = 3u;
            static constexpr uint32_t BytesS  = WavesM * 8192u; // per stage
            using TileF                       = lds::DimMajorTile<Cols, 64u>;
            static constexpr uint32_t BytesF  = TileF::bytes;
            static constexpr uint32_t CopiesF = TileF::copies / Waves;
            static constexpr uint32_t OutPitch = BlocksN * 64u + 16u; // bytes per row of a wave's results in LDS
            static constexpr uint32_t LdsBytes = RingS * BytesS + RingF * BytesF;
            static_assert(TileF::copies % Waves == 0u && (Waves * TileF::rowsPerCopy) % 16u == 0u, "whole copies per wave, swizzle periods");
            static_assert(Waves * 64u * OutPitch <= LdsBytes && LdsBytes <= Constants::AMDGCN_LDS_MAX_SIZE_BYTES, "LDS size");
        };

        // Byte offset of 16-byte piece `chunk` of row `row` in a 64 x 64 block of S.  The mask puts both readings of a
        // block on distinct banks: 16 lanes served together by a 16-byte read (rows with all values of bits 0..3, one chunk),
        // and the four rows times two 32-byte segments of a half-wave's transposing read.
        ROCWMMA_DEVICE inline uint32_t blockOffset(uint32_t row, uint32_t chunk)
        {
            const uint32_t mask = ((row >> 2) & 1u) | (((row >> 3) & 1u) << 1) | (((row >> 1) & 1u) << 2);
            return row * 128u + ((chunk ^ mask) << 4);
        }

        // f(integral_constant 0), f(1), ...: for bodies whose index must be a constant expression (instruction immediates)
        template <typename F, uint32_t... I>
        ROCWMMA_DEVICE ROCWMMA_INLINE void staticFor(std::integer_sequence<uint32_t, I...>, F&& f)
        {
            (f(std::integral_constant<uint32_t, I>{}), ...);
        }

        template <typename Cfg>
        __global__ void __launch_bounds__(Cfg::Threads) __attribute__((amdgpu_waves_per_eu(2, 2)))
            dlrmBwdTileKernel(const float16_t* input, const float16_t* upstream, float16_t* grad, float16_t* mlpGrad, uint32_t m, uint32_t k, uint32_t batch, uint32_t colTiles)
        {
            using FragF  = fragment<matrix_b, 32, 32, 16, float16_t, col_major>;
            using AccMap = detail::AccMap<32, 32, 32>;
            using TileF  = typename Cfg::TileF;
            constexpr uint32_t BN = Cfg::BlocksN, N = Cfg::Steps;
            extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];

            uint32_t sample, t;
            sampleAndTile(((m + Cfg::Rows - 1u) / Cfg::Rows) * colTiles, sample, t);
            if(sample >= batch) // (the whole workgroup)
                return;
            const uint32_t tid   = threadIdx.x;
            const uint32_t lane  = tid & 63u;
            const uint32_t wave  = __builtin_amdgcn_readfirstlane(tid >> 6);
            const uint32_t waveM = wave >> 1, waveN = wave & 1u;
            const uint32_t I0 = (t / colTiles) * Cfg::Rows, N0 = (t % colTiles) * Cfg::Cols;
            const uint32_t R0 = I0 + waveM * 64u; // this wave's rows

            const uint32_t   width = k + m * (m - 1u) / 2u; // (m <= 32768, k below 2^30: fits)
            const float16_t* feat  = input + static_cast<size_t>(sample) * m * k;
            const float16_t* up    = upstream + static_cast<size_t>(sample) * width;

            if(t == 0u) // bottom-MLP gradient = the first k entries of the upstream row
                for(uint32_t e = tid; e < k; e += Cfg::Threads)
                    mlpGrad[static_cast<size_t>(sample) * k + e] = up[e];

            const uint32_t stages = (m + 63u) / 64u;
            const uint32_t diag   = R0 / 64u; // the stage that meets this wave's part of the diagonal (or past the last)

            // ---- F: direct copies.  Rows from m on ask for an address past every sample and copy zeros (their offsets need not
            // fit 32 bits); columns from k on are whatever follows and only reach results that are never written.
            const uint32_t ldB   = k * 2u;
            const uint32_t lOffF = TileF::laneSourceOffset(lane, wave, ldB);
            const char*    fSrc  = reinterpret_cast<const char*>(feat) + N0 * 2u;
            const char*    fEnd  = reinterpret_cast<const char*>(feat + static_cast<size_t>(m) * k);
            uint32_t       rowsLeft = m;
            auto           copyF    = [&](uint32_t slot) {
                const lds::BufferRsrc src = lds::makeSource(fSrc, fEnd);
                char*                 to  = ldsRaw + Cfg::RingS * Cfg::BytesS + slot * Cfg::BytesF;
#pragma unroll
                for(uint32_t i = 0; i < Cfg::CopiesF; ++i)
                {
                    // (no branch around a copy: behind one the compiler waits for all that is in flight)
                    const uint32_t copy = i * Cfg::Waves + wave, row = copy * TileF::rowsPerCopy + lane / TileF::slotsPerRow;
                    lds::asyncCopy16(to + copy * 1024u, src, row < rowsLeft ? lOffF + TileF::copySourceOffset(copy, ldB) : kNowhere, 0u);
                }
                rowsLeft -= min(rowsLeft, 64u);
                fSrc += TileF::stageStep(ldB);
            };

            // ---- S: this wave carries 32 of its block's 64 rows, eight rows per load
            const uint32_t sRow   = waveN * 32u + (lane >> 3), sChunk = lane & 7u;
            // (row sRow + 8 i: 1024 bytes further per i, odd i flip the row's bit 3, i = 2, 3 set its bit 4)
            const uint32_t sStore = waveM * 8192u + blockOffset(sRow, sChunk), sStoreOdd = waveM * 8192u + blockOffset(sRow + 8u, sChunk) - 1024u;
            u32x4_t        rs[4], rs1[4]; // (the second only in front of the loop)
            // Byte offset in the upstream row of the entry a piece starts at: row hi, column lo, hi * (hi - 1) / 2 + lo entries behind
            // the first k.  From stage to stage the column moves by 64 below the diagonal; from the diagonal on the row does,
            // which is 64 * hi + 2016 entries.  A piece never runs past the end of its row except across the diagonal, and
            // there past the end of the sample at most: it then starts that much earlier (storeS), as do pieces of rows from
            // m on, which are cleared.
            uint32_t pieceAt[4], rowStep = 128u * (R0 + sRow) + 4032u;
            const uint32_t lastPiece = 2u * width - 16u;
#pragma unroll
            for(uint32_t i = 0; i < 4u; ++i)
            {
                const uint32_t hi = R0 + sRow + 8u * i;
                pieceAt[i]        = 2u * (k + hi * (hi - (hi != 0u)) / 2u + sChunk * 8u);
            }
            auto loadS = [&](u32x4_t(&rs)[4], uint32_t c0) {
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                    rs[i] = loadUnaligned(reinterpret_cast<const float16_t*>(reinterpret_cast<const char*>(up) + min(pieceAt[i], lastPiece)));
                const bool below = c0 < R0; // (wave uniform)
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                    pieceAt[i] += below ? 128u : rowStep + 1024u * i;
                rowStep += below ? 0u : 8192u;
                // Issued here, a stage ahead of their use: `upstream` is no __restrict pointer, or the compiler may move the
                // loads past this statement and past barriers.
                asm volatile("" ::: "memory");
            };
            auto storeS = [&](u32x4_t(&rs)[4], uint32_t c0) {
                const uint32_t first = max(R0, c0);
                if(first + 64u > m) // (wave uniform) rows from m on
                {
#pragma unroll
                    for(uint32_t i = 0; i < 4u; ++i)
                        if(first + sRow + 8u * i >= m)
                            rs[i] = u32x4_t{0u, 0u, 0u, 0u};
                }
                if(c0 == R0) // (wave uniform) across the diagonal: entries on and above it
                {
#pragma unroll
                    for(uint32_t i = 0; i < 4u; ++i)
                    {
                        // (a piece that starts `over` halves early is moved down by as many; past eight nothing of it is kept)
                        const uint32_t hi    = R0 + sRow + 8u * i;
                        const uint32_t start = k + hi * (hi - (hi != 0u)) / 2u + R0 + sChunk * 8u, over = start - min(start, width - 8u);
                        uint32_t       w[4]  = {rs[i][0], rs[i][1], rs[i][2], rs[i][3]};
                        const bool     two = (over & 4u) != 0u, one = (over & 2u) != 0u, half = (over & 1u) != 0u;
                        w[0] = two ? w[2] : w[0];
                        w[1] = two ? w[3] : w[1];
                        w[0] = one ? w[1] : w[0];
                        w[1] = one ? w[2] : w[1];
                        w[2] = one ? w[3] : w[2];
                        w[0] = half ? __builtin_amdgcn_alignbit(w[1], w[0], 16u) : w[0];
                        w[1] = half ? __builtin_amdgcn_alignbit(w[2], w[1], 16u) : w[1];
                        w[2] = half ? __builtin_amdgcn_alignbit(w[3], w[2], 16u) : w[2];
                        w[3] = half ? w[3] >> 16u : w[3];
                        const int keep = static_cast<int>(sRow + 8u * i) - static_cast<int>(sChunk * 8u); // entries in front of the diagonal
#pragma unroll
                        for(int j = 0; j < 4; ++j)
                            rs[i][j] = keep >= 2 * j + 2 ? w[j] : (keep == 2 * j + 1 ? w[j] & 0xFFFFu : 0u);
                    }
                }
                char* to = ldsRaw + ((c0 / 64u) % Cfg::RingS) * Cfg::BytesS;
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                    *reinterpret_cast<u32x4_t*>(to + ((i & 1u) ? sStoreOdd : sStore) + 1024u * i)
                        = (i & 2u) ? u32x4_t{rs[i][2], rs[i][3], rs[i][0], rs[i][1]} : rs[i];
            };

            // ---- fragments
            typedef short s16x4 __attribute__((ext_vector_type(4)));
            struct Frags
            {
                s16x4 a[2][2]; // [block of 32 rows][first / second four contraction indices of the lane's eight]
                FragF b[BN];
            };
            // Row by row: lane l reads row l % 32 of a block, piece 2 ks + l / 32, half by half.
            const uint32_t rowPart = waveM * 8192u + blockOffset(lane & 31u, lane >> 5) + ((lane >> 4) & 1u) * 8u;
            // Transposed: lane l gets row l % 32 of a block, contraction indices ks * 16 + (l / 32) * 8 + 0..7, as two transposing
            // reads: a group of 16 lanes gets the transpose of four rows of 32 bytes, eight bytes from each lane's address.
            const uint32_t grp = lane >> 4, s16 = lane & 15u;
            uint32_t       colPart[2][2]; // [block of 32 rows][first / second four contraction rows]
#pragma unroll
            for(uint32_t bi = 0; bi < 2u; ++bi)
#pragma unroll
                for(uint32_t kk = 0; kk < 2u; ++kk)
                    colPart[bi][kk] = waveM * 8192u + blockOffset((grp >> 1) * 8u + kk * 4u + (s16 >> 2), (bi * 2u + (grp & 1u)) * 2u + ((s16 & 3u) >> 1))
                                      + ((s16 & 1u) << 3);
            uint32_t fPart[BN];
#pragma unroll
            for(uint32_t j = 0; j < BN; ++j)
                fPart[j] = Cfg::RingS * Cfg::BytesS + TileF::offset((grp >> 1) * 8u + (s16 >> 2), waveN * BN * 2u + j * 2u + (grp & 1u)) + ((s16 & 3u) << 3);
            const uint32_t ldsBase = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds::LdsPtr)ldsRaw));
            // The two readings differ in their instruction, so the choice between them is a scalar branch inside one asm
            // statement: registers that reads in flight will write must not meet a branch the compiler sees (it could
            // move them there).  Across the diagonal both are read, waited for and joined (no bit is set in both: the
            // 64-bit addition is an OR).
            auto readS = [&](Frags& f, uint32_t stage, auto ksC) {
                constexpr uint32_t ks   = decltype(ksC)::value;
                const uint32_t     kind = __builtin_amdgcn_readfirstlane(stage < diag ? 0u : (stage == diag ? 1u : 2u));
                const uint32_t     base = ldsBase + (stage % Cfg::RingS) * Cfg::BytesS;
                const uint32_t     r    = base + (rowPart ^ (ks << 5));
                uint32_t           c[4];
#pragma unroll
                for(uint32_t j = 0; j < 4u; ++j)
                    c[j] = base + (colPart[j >> 1][j & 1u] ^ ((ks & 1u) << 3));
                s16x4              v0, v1, v2, v3, t0, t1;
                asm volatile("s_cmp_eq_u32 %[kind], 2\n\t"
                             "s_cbranch_scc1 .Labove%=\n\t"
                             "ds_read_b64 %[v0], %[r]\n\t"
                             "ds_read_b64 %[v2], %[r] offset:4096\n\t"
                             "ds_read_b64 %[v1], %[r8]\n\t"
                             "ds_read_b64 %[v3], %[r8] offset:4096\n\t"
                             "s_cmp_eq_u32 %[kind], 0\n\t"
                             "s_cbranch_scc1 .Ldone%=\n\t"
                             "ds_read_b64_tr_b16 %[t0], %[c0] offset:%[ks]\n\t"
                             "ds_read_b64_tr_b16 %[t1], %[c1] offset:%[ks]\n\t"
                             "s_waitcnt lgkmcnt(0)\n\t"
                             "v_lshl_add_u64 %[v0], %[t0], 0, %[v0]\n\t"
                             "v_lshl_add_u64 %[v1], %[t1], 0, %[v1]\n\t"
                             "ds_read_b64_tr_b16 %[t0], %[c2] offset:%[ks]\n\t"
                             "ds_read_b64_tr_b16 %[t1], %[c3] offset:%[ks]\n\t"
                             "s_waitcnt lgkmcnt(0)\n\t"
                             "v_lshl_add_u64 %[v2], %[t0], 0, %[v2]\n\t"
                             "v_lshl_add_u64 %[v3], %[t1], 0, %[v3]\n\t"
                             "s_branch .Ldone%=\n"
                             ".Labove%=:\n\t"
                             "ds_read_b64_tr_b16 %[v0], %[c0] offset:%[ks]\n\t"
                             "ds_read_b64_tr_b16 %[v1], %[c1] offset:%[ks]\n\t"
                             "ds_read_b64_tr_b16 %[v2], %[c2] offset:%[ks]\n\t"
                             "ds_read_b64_tr_b16 %[v3], %[c3] offset:%[ks]\n"
                             ".Ldone%=:"
                             : [v0] "=&v"(v0), [v1] "=&v"(v1), [v2] "=&v"(v2), [v3] "=&v"(v3), [t0] "=&v"(t0), [t1] "=&v"(t1)
                             : [kind] "s"(kind), [r] "v"(r), [r8] "v"(r ^ 8u), [c0] "v"(c[0]), [c1] "v"(c[1]), [c2] "v"(c[2]), [c3] "v"(c[3]),
                               [ks] "n"(ks * 2048u)
                             : "memory", "scc");
                f.a[0][0] = v0;
                f.a[0][1] = v1;
                f.a[1][0] = v2;
                f.a[1][1] = v3;
            };
            auto readStep = [&](Frags& f, uint32_t stage, uint32_t slotF, auto ksC) {
                constexpr uint32_t at   = decltype(ksC)::value * 16u * TileF::rowBytes;
                const uint32_t     base = ldsBase + slotF * Cfg::BytesF;
                readS(f, stage, ksC);
#pragma unroll
                for(uint32_t j = 0; j < BN; ++j)
                {
                    const uint32_t addr = base + fPart[j];
                    s16x4          v, w;
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(at) : "memory");
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(w) : "v"(addr), "n"(at + 4u * TileF::rowBytes) : "memory");
                    reinterpret_cast<s16x4*>(f.b[j].x)[0] = v;
                    reinterpret_cast<s16x4*>(f.b[j].x)[1] = w;
                }
            };
            auto pinFrags = [&](Frags& f) {
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                    lds::pinRegisters(f.a[i >> 1][i & 1u]);
#pragma unroll
                for(uint32_t j = 0; j < BN; ++j)
                    lds::pinRegisters(f.b[j].x);
            };

            FragAcc16 acc[2][BN];
#pragma unroll
            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                for(uint32_t j = 0; j < BN; ++j)
                    fill_fragment(acc[i][j], 0.0f);
            auto multiply = [&](Frags const& f) {
#pragma unroll
                for(uint32_t i = 0; i < 2u; ++i)
                {
                    FragK16 a;
                    reinterpret_cast<s16x4*>(a.x)[0] = f.a[i][0];
                    reinterpret_cast<s16x4*>(a.x)[1] = f.a[i][1];
#pragma unroll
                    for(uint32_t j = 0; j < BN; ++j)
                        mma_sync(acc[i][j], a, f.b[j], acc[i][j]);
                }
            };

            // ---- prologue: F(0 .. 2) and S(0 .. 2) all on their way together, S(0) and S(1) on to LDS
#pragma unroll
            for(uint32_t st = 0; st < Cfg::RingF; ++st)
                copyF(st);
            __builtin_amdgcn_sched_barrier(0);
            loadS(rs, 0u);
            loadS(rs1, 64u);
            __builtin_amdgcn_sched_barrier(0);
            storeS(rs, 0u);
            loadS(rs, 128u);
            __builtin_amdgcn_sched_barrier(0);
            storeS(rs1, 64u);
            lds::waitCopiesAndReads<2u * Cfg::CopiesF>(); // F(0) has landed
            lds::barrier();

            const std::integral_constant<uint32_t, 0u> first{};
            Frags                                      f[2];
            uint32_t                                   slotF = 0u; // of the stage that is multiplied
            readStep(f[0], 0u, 0u, first);
#pragma unroll 1
            for(uint32_t i = 0; i < stages; ++i)
            {
                staticFor(std::make_integer_sequence<uint32_t, N - 1u>{}, [&](auto ksC) {
                    constexpr uint32_t ks = decltype(ksC)::value;
                    lds::waitReads();
                    pinFrags(f[ks & 1u]);
                    __builtin_amdgcn_sched_barrier(0);
                    readStep(f[(ks + 1u) & 1u], i, slotF, std::integral_constant<uint32_t, ks + 1u>{});
                    multiply(f[ks & 1u]);
                    __builtin_amdgcn_sched_barrier(0);
                });
                // F(i + 1) has landed (F(i + 2) may be on its way), this wave's part of S(i + 1) is in LDS, stage i is in
                // registers.  The loads of S(i + 2) are not counted: into registers they may arrive in front of copies
                // into LDS that are older, so with them in the count a copy of F(i + 1) could be left out of it.
                lds::waitCopiesAndReads<Cfg::CopiesF>();
                pinFrags(f[(N - 1u) & 1u]);
                lds::barrier();
                __builtin_amdgcn_sched_barrier(0);
                copyF(slotF);
                slotF = slotF + 1u == Cfg::RingF ? 0u : slotF + 1u;
                readStep(f[0], i + 1u, slotF, first);
                __builtin_amdgcn_sched_barrier(0);
                storeS(rs, (i + 2u) * 64u);
                loadS(rs, (i + 3u) * 64u);
                multiply(f[(N - 1u) & 1u]);
                __builtin_amdgcn_sched_barrier(0);
            }
            // (the surplus copies still target this workgroup's LDS, the surplus reads these registers)
            lds::waitCopiesAndReads<0u>();
            pinFrags(f[0]);
            lds::barrier();

            // ---- results: this wave's rows through its own part of the LDS, then whole 16-byte pieces of rows
            char* mine = ldsRaw + wave * 64u * Cfg::OutPitch;
#pragma unroll
            for(uint32_t bi = 0; bi < 2u; ++bi)
#pragma unroll
                for(uint32_t j = 0; j < BN; ++j)
#pragma unroll
                    for(uint32_t r4 = 0; r4 < AccMap::runs; ++r4)
                    {
                        const uint32_t e0 = r4 * 4u;
                        float16_t      h[4];
#pragma unroll
                        for(uint32_t e = 0; e < 4u; ++e)
                            h[e] = static_cast<float16_t>(acc[bi][j].x[e0 + e]);
                        *reinterpret_cast<u32x2_t*>(mine + (bi * 32u + AccMap::rowOf(e0, lane)) * Cfg::OutPitch + (j * 32u + AccMap::colOf(e0, lane)) * 2u)
                            = *reinterpret_cast<u32x2_t*>(h);
                    }
            waveSync();
            constexpr uint32_t PerRow = BN * 4u; // 16-byte pieces
            const uint32_t     c      = N0 + waveN * BN * 32u + (lane % PerRow) * 8u;
            float16_t*         dst    = grad + static_cast<size_t>(sample) * m * k;
            if(c < k)
            {
#pragma unroll
                for(uint32_t rr = 0; rr < PerRow; ++rr)
                {
                    const uint32_t r = rr * (64u / PerRow) + lane / PerRow;
                    if(R0 + r < m)
                        *reinterpret_cast<u32x4_t*>(dst + static_cast<size_t>(R0 + r) * k + c)
                            = *reinterpret_cast<const u32x4_t*>(mine + r * Cfg::OutPitch + (lane % PerRow) * 16u);
                }
            }
        }

        // float32 backward through LDS.  32 contraction indices per stage; an instruction takes one float per lane,
        // so no transposing reads: "rows" as above (128 tile rows of 32 floats, 16-byte reads, instruction w of a
        // piece takes word w), "columns" = 32 contraction rows of 128 floats, row pitch 544 bytes (the two lane
        // halves of an instruction read rows four apart: 4 x 544 bytes puts them on different banks), 4-byte reads.
        constexpr uint32_t kStageK32   = 32;
        constexpr uint32_t kColPitch32 = 544;
        constexpr uint32_t kColsBytes32 = kStageK32 * kColPitch32; // 17408

        __global__ void __launch_bounds__(256, 3) dlrmBwdStagedF32Kernel(const float* __restrict__ input,
                                                                         const float* __restrict__ upstream,
                                                                         float* __restrict__ grad,
                                                                         float* __restrict__ mlpGrad,
                                                                         uint32_t m,
                                                                         uint32_t k,
                                                                         uint32_t batch,
                                                                         uint32_t colTiles)
        {
            using FragS   = fragment<matrix_a, 32, 32, 2, float32_t, row_major>;
            using FragF   = fragment<matrix_b, 32, 32, 2, float32_t, row_major>;
            using FragAcc = fragment<accumulator, 32, 32, 2, float32_t>;
            using AccMap  = detail::AccMap<32, 32, 32>;

            __shared__ __attribute__((aligned(16))) char ldsS[kRowsBytes]; // "rows" or "columns" layout, by stage
            __shared__ __attribute__((aligned(16))) char ldsF[kColsBytes32]; // "columns" layout

            uint32_t sample, t;
            sampleAndTile(((m + kTile - 1u) / kTile) * colTiles, sample, t);
            if(sample >= batch) // (the whole workgroup)
                return;
            const uint32_t tid  = threadIdx.x;
            const uint32_t lane = tid & 63u;
            const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const uint32_t I = t / colTiles, N = t % colTiles;
            const uint32_t I0 = I * kTile, N0 = N * kTile;

            const size_t width = packedRow(k, m);
            const float* feat  = input + static_cast<size_t>(sample) * m * k;
            const float* up    = upstream + static_cast<size_t>(sample) * width;
            float*       dst   = grad + static_cast<size_t>(sample) * m * k;

            if(t == 0u) // bottom-MLP gradient = the first k entries of the upstream row
                for(uint32_t e = tid; e < k; e += 256u)
                    mlpGrad[static_cast<size_t>(sample) * k + e] = up[e];

            const uint32_t wr = wave >> 1, wc = wave & 1u;
            const bool     waveLive = I0 + wr * kWaveTile < m && N0 + wc * kWaveTile < k; // (every wave stages and meets the barriers)

            // (as in the float16 kernel) where a stage lies against the tile's rows decides how S arrives
            enum Where : uint32_t { Below, Above, Across };
            auto whereOf = [&](uint32_t c0) { return c0 + kStageK32 <= I0 ? Below : (c0 >= I0 + kTile ? Above : Across); };

            // this thread's pieces.  "rows": tile rows tid / 8 + 32 i, piece tid % 8; "columns": contraction rows
            // tid / 32 + 8 i, piece tid % 32.
            const lds::BufferRsrc rsrcF = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(feat), 0, static_cast<int>(m * k * 4u), 0x00020000);
            const uint32_t        posR = tid & 7u, posC = tid & 31u;
            const bool            colInK = N0 + posC * 4u < k;
            size_t                belowStart[4];
#pragma unroll
            for(uint32_t i = 0; i < 4u; ++i)
                belowStart[i] = packedRow(k, min(I0 + (tid >> 3) + 32u * i, m - 1u));

            u32x4_t rs[4], rf[4];
            auto    fetch = [&](uint32_t c0) { // (c0 < m)
                const Where where = whereOf(c0);
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                {
                    const uint32_t cr = (tid >> 5) + 8u * i;
                    rf[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrcF, static_cast<int>(colInK ? (min(c0 + cr, m) * k + N0 + posC * 4u) * 4u : kNowhere), 0, 0);
                    // (rows of the packed triangle start at any float: 4-byte aligned 16-byte loads)
                    if(where == Below)
                        rs[i] = *reinterpret_cast<const u32x4_t __attribute__((aligned(4)))*>(up + belowStart[i] + c0 + posR * 4u);
                    else if(where == Above)
                        rs[i] = *reinterpret_cast<const u32x4_t __attribute__((aligned(4)))*>(up + packedRow(k, min(c0 + cr, m - 1u)) + I0 + posC * 4u);
                }
            };

            FragAcc acc[2][2];
#pragma unroll
            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                for(uint32_t j = 0; j < 2u; ++j)
                    fill_fragment(acc[i][j], 0.0f);

            const uint32_t row = lane & 31u, half = lane >> 5;
            fetch(0u);
#pragma unroll 1
            for(uint32_t c0 = 0; c0 < m; c0 += kStageK32)
            {
                const Where where = whereOf(c0);
#pragma unroll
                for(uint32_t i = 0; i < 4u; ++i)
                {
                    const uint32_t cr = (tid >> 5) + 8u * i;
                    *reinterpret_cast<u32x4_t*>(ldsF + cr * kColPitch32 + posC * 16u) = rf[i];
                    if(where == Below)
                        *reinterpret_cast<u32x4_t*>(ldsS + ((tid >> 3) + 32u * i) * kRowPitch + posR * 16u) = rs[i];
                    else if(where == Above)
                        *reinterpret_cast<u32x4_t*>(ldsS + cr * kColPitch32 + posC * 16u) = c0 + cr < m ? rs[i] : u32x4_t{0u, 0u, 0u, 0u};
                }
                if(where == Across)
                {
#pragma unroll 4
                    for(uint32_t i = 0; i < 16u; ++i)
                    {
                        const uint32_t r  = (tid >> 5) + 8u * i, c = tid & 31u;
                        const uint32_t Rg = I0 + r, cg = c0 + c;
                        const uint32_t hi = Rg > cg ? Rg : cg, lo = Rg > cg ? cg : Rg;
                        float          v  = 0.0f;
                        if(hi < m && Rg != cg)
                            v = up[packedRow(k, hi) + lo];
                        *reinterpret_cast<float*>(ldsS + r * kRowPitch + c * 4u) = v;
                    }
                }
                __syncthreads();
                if(c0 + kStageK32 < m)
                    fetch(c0 + kStageK32);
                __builtin_amdgcn_sched_barrier(0);
                if(waveLive)
                {
                    // instruction (ks, w) contracts c = ks * 8 + half * 4 + w of the stage
#pragma unroll
                    for(uint32_t ks = 0; ks < 4u; ++ks)
                    {
                        u32x4_t sp[2];
                        if(where != Above)
                        {
#pragma unroll
                            for(uint32_t i = 0; i < 2u; ++i)
                                sp[i] = rowsFragment(ldsS, wr * 2u + i, ks, lane);
                        }
#pragma unroll
                        for(uint32_t w = 0; w < 4u; ++w)
                        {
                            const uint32_t cr = ks * 8u + half * 4u + w;
                            FragS          a[2];
                            FragF          b[2];
#pragma unroll
                            for(uint32_t j = 0; j < 2u; ++j)
                                b[j].x[0] = *reinterpret_cast<const float*>(ldsF + cr * kColPitch32 + ((wc * 2u + j) * 32u + row) * 4u);
                            if(where == Above)
                            {
#pragma unroll
                                for(uint32_t i = 0; i < 2u; ++i)
                                    a[i].x[0] = *reinterpret_cast<const float*>(ldsS + cr * kColPitch32 + ((wr * 2u + i) * 32u + row) * 4u);
                            }
                            else
                            {
#pragma unroll
                                for(uint32_t i = 0; i < 2u; ++i)
                                    a[i] = pieceFragment<FragS>(sp[i], w);
                            }
#pragma unroll
                            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                                for(uint32_t j = 0; j < 2u; ++j)
                                    mma_sync(acc[i][j], a[i], b[j], acc[i][j]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
            }

            if(!waveLive)
                return;
            // a lane owns runs of four consecutive columns of one row (k is a multiple of 4)
#pragma unroll
            for(uint32_t i = 0; i < 2u; ++i)
#pragma unroll
                for(uint32_t j = 0; j < 2u; ++j)
#pragma unroll
                    for(uint32_t r4 = 0; r4 < AccMap::runs; ++r4)
                    {
                        const uint32_t e0 = r4 * 4u;
                        const uint32_t r  = I0 + wr * kWaveTile + i * 32u + AccMap::rowOf(e0, lane);
                        const uint32_t c  = N0 + wc * kWaveTile + j * 32u + AccMap::colOf(e0, lane);
                        if(r < m && c < k)
                            *reinterpret_cast<f32x4_t*>(dst + static_cast<size_t>(r) * k + c)
                                = f32x4_t{acc[i][j].x[e0], acc[i][j].x[e0 + 1u], acc[i][j].x[e0 + 2u], acc[i][j].x[e0 + 3u]};
                    }
        }

        // workgroups of a launch (see sampleAndTile), 0 if they do not fit a grid dimension
        inline uint32_t gridFor(uint32_t tiles, uint32_t batch)
        {
            const uint64_t workgroups = static_cast<uint64_t>((batch + kXcds - 1u) / kXcds) * kXcds * tiles;
            return workgroups <= 0x7FFFFFFFull ? static_cast<uint32_t>(workgroups) : 0u;
        }

        template <typename Cfg>
        int launchBwdTile(const void* input, const void* upstream, void* grad, void* mlpGrad, uint32_t m, uint32_t k, uint32_t batch,
                          hipStream_t stream)
        {
            const uint32_t rowTiles = (m + Cfg::Rows - 1u) / Cfg::Rows, colTiles = (k + Cfg::Cols - 1u) / Cfg::Cols;
            if(static_cast<uint64_t>(rowTiles) * colTiles > 0x7FFFFFFFull)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            const uint32_t grid = gridFor(rowTiles * colTiles, batch);
            if(grid == 0u)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            auto kernel = dlrmBwdTileKernel<Cfg>;
            // more than 64 KiB of dynamic LDS needs an explicit opt-in (idempotent, no allocation)
            if(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(Cfg::LdsBytes))
               != hipSuccess)
                return ROCWMMA_AMD_LAUNCH_FAILED;
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::Threads), Cfg::LdsBytes, stream, static_cast<const float16_t*>(input),
                               static_cast<const float16_t*>(upstream), static_cast<float16_t*>(grad), static_cast<float16_t*>(mlpGrad), m,
                               k, batch, colTiles);
            return launchStatus();
        }

        // Which tile: the one with the less estimated time, from timings of both at 25 shapes (m 129 to 4096, k 8 to 1024, batch
        // 9 to 64).  A round of 256 x 256 tiles, one per compute unit, takes 7 us plus 2.05 per stage; 128 x 128 tiles run two per
        // unit, 3 plus 1.55 per stage for the two, and a lone one 4 plus 0.7.  Large / small in us: (1024, 1024, 64) 185 / 224,
        // (512, 1024, 32) 28 / 34, (129, 1024, 33) 12.5 / 14; (360, 256, 32) 17 / 11, (900, 64, 64) 39 / 32, (600, 600, 64) 78 / 72.
        int launchBwdF16(const void* input, const void* upstream, void* grad, void* mlpGrad, uint32_t m, uint32_t k, uint32_t batch,
                         hipStream_t stream)
        {
            using Large = BwdTile<4, 4>;
            using Small = BwdTile<2, 2>;
            const float    stages = static_cast<float>((m + 63u) / 64u);
            const uint64_t units  = computeUnits();
            const uint64_t large  = static_cast<uint64_t>((m + 255u) / 256u) * ((k + 255u) / 256u) * batch;
            const uint64_t small  = static_cast<uint64_t>((m + 127u) / 128u) * ((k + 127u) / 128u) * batch;
            const float    tLarge = static_cast<float>((large + units - 1u) / units) * (7.0f + 2.05f * stages) + 1.0f;
            const float    tSmall = small <= units ? 7.0f + 0.7f * stages
                                                   : static_cast<float>((small + 2u * units - 1u) / (2u * units)) * (3.0f + 1.55f * stages) + 3.0f;
            return tLarge < tSmall ? launchBwdTile<Large>(input, upstream, grad, mlpGrad, m, k, batch, stream)
                                   : launchBwdTile<Small>(input, upstream, grad, mlpGrad, m, k, batch, stream);
        }
    } // namespace

    namespace
    {
        // float16 forward, where dlrmFwdStagedKernel is ahead of the tiles of dlrm_general_fwd.hip: batches of many rounds of tiles (two
        // per unit) whose tiles are partly filled or half above the diagonal.  Its waves skip 64 x 64 blocks that hold no result
        // and four of its workgroups share a unit.  Staged / tiles in us: (193, 64) batch 4096 118 / 128, (256, 64) 145 / 163,
        // (320, 128) 32 rounds 1.16 times, (400, 128) 451 / 481; but 8 rounds of (256, 128) 0.97, (384, k) never above 1.02, (512, k) 0.80
        // to 0.99.  One tile per sample (up to 128 rows that do not fit the LDS): (96, 512) batch 1024 26.3.
        bool stagedFwdIsFaster(uint32_t m, uint32_t k, uint32_t tiles, uint32_t batch)
        {
            const uint64_t units = computeUnits(), rounds = static_cast<uint64_t>(tiles) * batch / (2u * units);
            if(m <= 128u)
                return batch > units;
            if(m <= 256u)
                return k <= 512u && rounds >= 12u;
            if(m <= 352u)
                return k <= 512u && rounds >= 6u;
            return m > 384u && m <= 416u && k <= 256u && rounds >= 24u;
        }
    } // namespace

    // Shapes: 1 <= m <= 32768; k a multiple of 8 (f16) or 4 (f32), so that a row's 16-byte pieces are whole; a sample's
    // features below 2 GiB (32-bit byte offsets into a bounds-checked buffer).
    int launchDlrmFwdGeneral(int dtype, const void* input, void* output, uint32_t m, uint32_t k, uint32_t batch, hipStream_t stream)
    {
        const uint32_t size = dtype == ROCWMMA_AMD_F16 ? 2u : 4u;
        if(m > kMaxRows || k == 0u || k % (16u / size) != 0u || static_cast<uint64_t>(m) * k * size >= (1ull << 31))
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t side = (m + kTile - 1u) / kTile, tiles = side * (side + 1u) / 2u;
        const uint32_t grid = gridFor(tiles, batch);
        if(grid == 0u)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        if(dtype == ROCWMMA_AMD_F16)
        {
            const int rc = stagedFwdIsFaster(m, k, tiles, batch) ? ROCWMMA_AMD_UNSUPPORTED_SHAPE : launchDlrmFwdTilesF16(input, output, m, k, batch, stream);
            if(rc != ROCWMMA_AMD_UNSUPPORTED_SHAPE) // (feature rows of more than 16 MiB)
                return rc;
            hipLaunchKernelGGL(dlrmFwdStagedKernel<float16_t>, dim3(grid), dim3(256), 0, stream, static_cast<const float16_t*>(input),
                               static_cast<float16_t*>(output), m, k, batch, tiles);
        }
        else
            hipLaunchKernelGGL(dlrmFwdStagedKernel<float>, dim3(grid), dim3(256), 0, stream, static_cast<const float*>(input),
                               static_cast<float*>(output), m, k, batch, tiles);
        return launchStatus();
    }

    int launchDlrmBwdGeneral(int dtype, const void* input, const void* upstream, void* grad, void* mlpGrad, uint32_t m, uint32_t k,
                             uint32_t batch, hipStream_t stream)
    {
        const uint32_t size = dtype == ROCWMMA_AMD_F16 ? 2u : 4u;
        if(m > kMaxRows || k == 0u || k % (16u / size) != 0u || static_cast<uint64_t>(m) * k * size >= (1ull << 31))
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t rowTiles = (m + kTile - 1u) / kTile, colTiles = (k + kTile - 1u) / kTile;
        if(static_cast<uint64_t>(rowTiles) * colTiles > 0x7FFFFFFFull)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t grid = gridFor(rowTiles * colTiles, batch);
        if(grid == 0u)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        if(dtype == ROCWMMA_AMD_F16)
            return launchBwdF16(input, upstream, grad, mlpGrad, m, k, batch, stream);
        hipLaunchKernelGGL(dlrmBwdStagedF32Kernel, dim3(grid), dim3(256), 0, stream, static_cast<const float*>(input),
                               static_cast<const float*>(upstream), static_cast<float*>(grad), static_cast<float*>(mlpGrad), m, k, batch,
                               colTiles);
        return launchStatus();
    }
} // namespace rocwmma_amd
