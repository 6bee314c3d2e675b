// GEMM with few results for its K (few token rows against a weight matrix above all): D = act(alpha * A * B + beta * C + bias), A
// row-major, B col-major, C / D row-major, any K.  Included by the translation units that instantiate it.
//
// The reference's GEMM kernels (samples/perf_hgemm.cpp:518-714) and the blocked kernel here give a workgroup a tile of D and all
// of K: with few rows and columns there are few tiles, each walks K alone, and most of the chip idles.  Here the waves of a workgroup
// share K instead: MB blocks of 16 rows of A and NB of 16 weight rows per workgroup, and every wave multiplies a quarter or an
// eighth of K of all of them.  Its operands come through a ring of 128-byte steps in LDS that is the wave's own, so the main loop
// has no barrier.  (Fragments loaded straight into registers were two to three times slower: the 16 lanes that a load serves
// together are 16 rows, i.e. 16 lines for 256 bytes, 30 GB/s per compute unit; a copy into LDS takes whole lines.)  The
// partial sums meet in LDS and are added in the order of the waves: results do not depend on timing.  What bounds it is a
// compute unit's copies: (MB + NB) * 16 rows of K for NB * 16 columns of results, about 100 GB/s of them by one unit and 12 TB/s by
// all.  Before (blocked or weight-streaming kernel) and now, us: 16 x 3056 x 7168 bf16 with GELU 39.2 -> 11.8, 16 x 1776 x 5824 f16
// 28.5 -> 7.2, 64 x 1024 x 8192 f16 30.3 -> 14.9, 32 x 2848 x 6656 int8 16.7 -> 6.5, 416 x 480 x 5280 f16 25.3 -> 15.4,
// 112 x 320 x 5632 f16 23.5 -> 6.7, 240 x 592 x 2240 bf16 12.2 -> 6.4.
#ifndef ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_HPP
#define ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_HPP

#include "common.hpp"
#include "gemm_few_rows_rule.hpp"
#include <utility>
#include <rocwmma/rocwmma_lds.hpp>

using namespace rocwmma;

namespace rocwmma_amd
{
    namespace
    {
        constexpr uint32_t kFewXcds    = 8u; // dies, one L2 each
        constexpr uint32_t kFewNowhere = 0x80000000u; // lane offset beyond every buffer: the load returns zeros

        template <uint32_t MB_, uint32_t NB_>
        struct FewTile
        {
            static constexpr uint32_t MB = MB_, NB = NB_; // blocks of 16 rows of A, of 16 weight rows
            static constexpr uint32_t Waves = fewWaves(MB, NB), Ring = fewRing(MB, NB);
            static constexpr uint32_t StepBytes = (MB + NB) * 16u * kFewStep, Copies = StepBytes / 1024u;
            static constexpr uint32_t LdsBytes = Waves * Ring * StepBytes;
            static_assert(kFewLds == Constants::AMDGCN_LDS_MAX_SIZE_BYTES && Ring >= 2u && (Ring - 1u) * Copies < 64u && Waves * MB * NB * 1024u <= LdsBytes, "ring and partial sums in LDS");
        };

        template <typename InT, typename OutT, typename CompT, typename Tile>
        __global__ void __launch_bounds__(64u * Tile::Waves) gemmFewRowsKernel(GemmArgs g)
        {
            constexpr uint32_t E = sizeof(InT), MB = Tile::MB, NB = Tile::NB, Waves = Tile::Waves, Ring = Tile::Ring;
            constexpr uint32_t K = kFewStep / E;
            using FragA          = fragment<matrix_a, 16, 16, K, InT, row_major>;
            using FragB          = fragment<matrix_b, 16, 16, K, InT, col_major>;
            using FragAcc        = fragment<accumulator, 16, 16, K, CompT>;
            using Rows           = lds::KMajorTile<16u, kFewStep>; // 16 rows of one step
            using Quad           = CompT __attribute__((ext_vector_type(4)));
            static_assert(sizeof(FragA::x) == 32u && sizeof(FragB::x) == 32u, "a step is two pieces of 16 bytes per lane");
            extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];

            const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            const uint32_t row = lane & 15u, group = lane >> 4; // of a lane's results in a block: its row, its four columns
            // Workgroups of the same weights on one XCD (ids congruent mod 8), whose L2 then fetches them once.
            const uint32_t groupsM = ceilDiv(g.m, MB * 16u), id = blockIdx.x / kFewXcds;
            const uint32_t m0 = id % groupsM * MB * 16u, n0 = (id / groupsM * kFewXcds + blockIdx.x % kFewXcds) * NB * 16u;
            if(n0 >= g.n) // (the whole workgroup)
                return;
            const uint32_t ldaB = g.lda * E, ldbB = g.ldb * E, kBytes = g.k * E;
            const uint32_t steps = ceilDiv(kBytes, kFewStep), begin = steps * wave / Waves, end = steps * (wave + 1u) / Waves;
            const uint32_t kEnd = min(kBytes, end * kFewStep); // this wave's part of K ends here

            // Copies of eight rows.  Lanes past the part's end, and blocks past the last row of A or B, ask for an address beyond the
            // buffer and copy zeros.
            uint32_t laneK[2], aOff[2], bOff[2];
#pragma unroll
            for(uint32_t half = 0; half < 2u; ++half)
            {
                laneK[half] = Rows::laneK(lane, half);
                aOff[half]  = Rows::laneSourceOffset(lane, half, ldaB);
                bOff[half]  = Rows::laneSourceOffset(lane, half, ldbB);
            }
            const lds::BufferRsrc srcA = lds::makeSource(static_cast<const char*>(g.a) + static_cast<size_t>(m0) * ldaB);
            const lds::BufferRsrc srcB = lds::makeSource(static_cast<const char*>(g.b) + static_cast<size_t>(n0) * ldbB);
            char* const           ring = ldsRaw + wave * (Ring * Tile::StepBytes);
            auto                  issue = [&](uint32_t slot, uint32_t step) {
                char* const    to = ring + slot * Tile::StepBytes;
                // (readfirstlane: the 64 x 32 tile had the copies' offsets in vector registers, and every copy was a loop over the lanes')
                const uint32_t at = __builtin_amdgcn_readfirstlane(step * kFewStep);
                uint32_t       a[2], b[2];
#pragma unroll
                for(uint32_t half = 0; half < 2u; ++half)
                {
                    const bool inside = laneK[half] + at < kEnd;
                    a[half]           = inside ? aOff[half] : kFewNowhere;
                    b[half]           = inside ? bOff[half] : kFewNowhere;
                }
#pragma unroll
                for(uint32_t c = 0; c < 2u * NB; ++c)
                    lds::asyncCopy16(to + (2u * MB + c) * 1024u, srcB, n0 + c / 2u * 16u < g.n ? b[c % 2u] : kFewNowhere, c * 8u * ldbB + at);
#pragma unroll
                for(uint32_t c = 0; c < 2u * MB; ++c)
                    lds::asyncCopy16(to + c * 1024u, srcA, m0 + c / 2u * 16u < g.m ? a[c % 2u] : kFewNowhere, c * 8u * ldaB + at);
            };

            FragAcc acc[MB][NB];
#pragma unroll
            for(uint32_t i = 0; i < MB; ++i)
#pragma unroll
                for(uint32_t j = 0; j < NB; ++j)
                    fill_fragment(acc[i][j], static_cast<CompT>(0));

#pragma unroll
            for(uint32_t u = 0; u < Ring; ++u)
                issue(u, begin + u);
            uint32_t slot = 0u;
#pragma unroll 1
            for(uint32_t s = begin; s < end; ++s)
            {
                lds::waitCopiesAndReads<(Ring - 1u) * Tile::Copies>(); // step s has landed
                asm volatile("" ::: "memory");
                const char* from = ring + slot * Tile::StepBytes;
                FragA       a[MB];
                FragB       b[NB];
#pragma unroll
                for(uint32_t p = 0; p < 2u; ++p)
                {
#pragma unroll
                    for(uint32_t j = 0; j < NB; ++j)
                        Rows::template readBlock16<16u>(reinterpret_cast<char*>(b[j].x) + 16u * p, from + (MB + j) * Rows::bytes, 0u, p, lane);
#pragma unroll
                    for(uint32_t i = 0; i < MB; ++i)
                        Rows::template readBlock16<16u>(reinterpret_cast<char*>(a[i].x) + 16u * p, from + i * Rows::bytes, 0u, p, lane);
                }
                lds::waitReads(); // the slot is free
                asm volatile("" ::: "memory");
                issue(slot, s + Ring);
                slot = slot + 1u == Ring ? 0u : slot + 1u;
#pragma unroll
                for(uint32_t i = 0; i < MB; ++i)
#pragma unroll
                    for(uint32_t j = 0; j < NB; ++j)
                        mma_sync(acc[i][j], a[i], b[j], acc[i][j]);
            }
            lds::waitCopiesAndReads<0u>(); // the surplus copies still target the ring, where the partial sums go next
            __syncthreads();

            // The partial sums: wave w's of block b at [w][b][lane], a lane's four results (row lane % 16, columns 4 (lane / 16) ..)
            Quad* partial = reinterpret_cast<Quad*>(ldsRaw);
#pragma unroll
            for(uint32_t i = 0; i < MB; ++i)
#pragma unroll
                for(uint32_t j = 0; j < NB; ++j)
                    partial[((wave * MB + i) * NB + j) * 64u + lane] = *reinterpret_cast<Quad*>(acc[i][j].x);
            __syncthreads();
            for(uint32_t block = wave; block < MB * NB; block += Waves)
            {
                const uint32_t r = m0 + block / NB * 16u + row, col = n0 + block % NB * 16u + group * 4u;
                Quad           sum = partial[block * 64u + lane];
#pragma unroll
                for(uint32_t w = 1; w < Waves; ++w)
                    sum += partial[(w * MB * NB + block) * 64u + lane];
                if(r >= g.m || col >= g.n)
                    continue;
                const CompT alpha = static_cast<CompT>(g.alpha), beta = static_cast<CompT>(g.beta);
                typedef uint32_t Words __attribute__((ext_vector_type(sizeof(OutT))));
                CompT            v[4];
                OutT             o[4];
#pragma unroll
                for(uint32_t e = 0; e < 4u; ++e)
                    v[e] = alpha * sum[e];
                if(beta != static_cast<CompT>(0))
                {
                    const Words w = *reinterpret_cast<const Words*>(static_cast<const OutT*>(g.c) + static_cast<size_t>(r) * g.ldc + col);
                    __builtin_memcpy(o, &w, sizeof(w));
#pragma unroll
                    for(uint32_t e = 0; e < 4u; ++e)
                        v[e] += beta * static_cast<CompT>(o[e]);
                }
                if constexpr(std::is_same<CompT, float>::value)
                {
                    if(g.bias)
                    {
#pragma unroll
                        for(uint32_t e = 0; e < 4u; ++e)
                            v[e] += g.bias[col + e];
                    }
                    applyActivation(v, g.activation);
                }
#pragma unroll
                for(uint32_t e = 0; e < 4u; ++e)
                    o[e] = narrowed<OutT>(v[e]);
                Words w;
                __builtin_memcpy(&w, o, sizeof(w));
                *reinterpret_cast<Words*>(static_cast<OutT*>(g.d) + static_cast<size_t>(r) * g.ldd + col) = w;
            }
        }

        // f(integral_constant 0), f(1), ...
        template <typename F, uint32_t... I>
        void forTiles(F& f, std::integer_sequence<uint32_t, I...>)
        {
            (f(std::integral_constant<uint32_t, I>{}), ...);
        }

        template <typename InT, typename OutT, typename CompT, uint32_t MB, uint32_t NB>
        int launchFewTile(GemmArgs const& g, hipStream_t stream)
        {
            using Tile  = FewTile<MB, NB>;
            auto kernel = gemmFewRowsKernel<InT, OutT, CompT, Tile>;
            if(Tile::LdsBytes > 65536u
               && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(Tile::LdsBytes))
                      != hipSuccess)
                return ROCWMMA_AMD_LAUNCH_FAILED;
            hipLaunchKernelGGL(kernel, dim3(ceilDiv(g.m, MB * 16u) * ceilDiv(g.n, NB * 16u * kFewXcds) * kFewXcds), dim3(64u * Tile::Waves), Tile::LdsBytes, stream, g);
            return launchStatus();
        }

        template <typename InT, typename OutT, typename CompT>
        int launchFewRows(GemmArgs const& g, hipStream_t stream, FewChoice const& choice)
        {
            // (copies address a workgroup's rows of A, and its weights, inside a 2 GiB window)
            if(static_cast<uint64_t>(g.lda) * sizeof(InT) * 16u * choice.mb >= 0x7FFF0000ull
               || static_cast<uint64_t>(g.ldb) * sizeof(InT) * 16u * choice.nb >= 0x7FFF0000ull)
                return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            int  rc      = ROCWMMA_AMD_UNSUPPORTED_SHAPE;
            auto attempt = [&](auto index) {
                constexpr FewCost tile = kFewCosts[decltype(index)::value];
                if(tile.mb == choice.mb && tile.nb == choice.nb)
                    rc = launchFewTile<InT, OutT, CompT, tile.mb, tile.nb>(g, stream);
            };
            forTiles(attempt, std::make_integer_sequence<uint32_t, kFewTiles>{});
            return rc;
        }
    } // namespace
} // namespace rocwmma_amd

#endif // ROCWMMA_AMD_CSRC_GEMM_FEW_ROWS_HPP
