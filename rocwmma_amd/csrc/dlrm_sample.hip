// DLRM dot interaction for samples of up to 192 feature rows and any width of whole 16-byte pieces that fit the LDS,
// float16 and float32; semantics = dlrm_fwd_CPU / dlrm_bwd_CPU (test/reference_impl.hpp:83-179).
//
// A sample is the work of one, two, four or eight waves.  Its feature rows (backward: and its upstream row) go to LDS
// once, as whole-wave 1 KiB direct copies, all in flight together (a lane per 16 bytes; lanes that fall on the row
// pitch or on the row of zeros behind the last feature row ask for an address beyond the sample and store zeros),
// and both matrix operands are read from there:
//
//   * 16 x 16 blocks (v_mfma_f32_16x16x32_f16, v_mfma_f32_16x16x4_f32): 41 rows are 3 blocks of 16, six products for
//     the lower triangle, where 128 x 128 tiles multiplied 16384 entries for 820;
//   * rows past m and pieces past k read the row of zeros, so m and k are run-time values and nothing of a
//     neighbouring sample can leak (0 * Inf);
//   * the row pitch is an odd number of 16-byte pieces: the 16 rows of a fragment read fall into 16 bank groups;
//   * forward: a wave keeps its blocks of the lower triangle in registers until all waves have read the features, then
//     the packed triangle takes their place in LDS and leaves in 16-byte pieces;
//   * backward: a G fragment (16 rows of the symmetric matrix) is gathered from the packed triangle in LDS and kept for
//     every column of its rows; gradient rows leave the accumulators as 64 contiguous bytes per row (float16 after
//     exchanging halves between neighbouring 16-lane rows).
//
// Bound by memory where the batch fills the device; forward + backward, against one wave per sample with operands straight
// from global memory (float32) or two waves per workgroup (float16, 33 to 128 rows) or 128 x 128 tiles (other widths):
// 27 x 128 float32 batch 65536 764 -> 557 us (5.4 TB/s), 45 x 128 float16 batch 13033 139 -> 93 us, 41 x 72 float16 batch
// 8192 119 -> 41 us (4.3 TB/s), 94 x 232 float16 batch 5738 394 -> 183 us.  (A first version unpacked G into an LDS
// square with loads of its own, a serial chain of load latencies: 41 x 72 backward 65 instead of 26 us.)
#include "common.hpp"
#include "launch_limits.hpp"
#include <rocwmma/rocwmma_lds.hpp>

using namespace rocwmma;

namespace rocwmma_amd
{
    namespace
    {
        typedef uint32_t u32x4_t __attribute__((ext_vector_type(4), may_alias));
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2), may_alias));
        typedef float    f32x4_t __attribute__((ext_vector_type(4)));
        typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
        typedef short    s16x4_t __attribute__((ext_vector_type(4)));

        constexpr uint32_t wavesOf(uint32_t perSample) // per workgroup
        {
            return perSample > 4u ? perSample : 4u;
        }
        constexpr uint32_t kNowhere  = 0x80000000u; // beyond every sample: a bounds-checked copy from there stores zeros
        constexpr uint32_t kLdsBytes = 160u * 1024u;
        constexpr uint32_t kMaxRows  = 192;

        // Geometry of a sample in LDS, the same for every workgroup of a launch.
        struct SampleShape
        {
            uint32_t m, k, batch;
            uint32_t pieces; // 16-byte pieces of a feature row
            uint32_t pitch; // LDS row pitch in pieces (odd)
            uint32_t pitchMagic; // ceil(2^32 / pitch): piece / pitch as a multiplication
            uint32_t featBytes; // feature rows and the row of zeros, whole copies
            uint32_t sampleBytes; // LDS per sample
            uint32_t width; // of a packed row
        };

        ROCWMMA_DEVICE inline void waveSync()
        {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        // all waves of a sample (a single wave needs no barrier: the LDS serves its accesses in order)
        template <uint32_t PerSample>
        ROCWMMA_DEVICE inline void sampleSync()
        {
            if constexpr(PerSample == 1u)
                waveSync();
            else
                __syncthreads();
        }

        // This wave's share of the copies of a sample's rows into `tile`.
        template <uint32_t PerSample>
        ROCWMMA_DEVICE inline void loadFeatures(char* tile, const void* features, SampleShape const& s, uint32_t part, uint32_t lane)
        {
            const uint32_t        bytes = s.m * s.pieces * 16u;
            const lds::BufferRsrc rsrc  = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(features), 0, static_cast<int>(bytes), 0x00020000);
            for(uint32_t copy = part; copy * 1024u < s.featBytes; copy += PerSample)
            {
                const uint32_t piece = copy * 64u + lane;
                const uint32_t row   = __umulhi(piece, s.pitchMagic);
                const uint32_t pos   = piece - row * s.pitch;
                lds::asyncCopy16Streaming(tile + copy * 1024u, rsrc, pos < s.pieces ? (row * s.pieces + pos) * 16u : kNowhere, 0u);
            }
        }

        // Rows of a 16-row fragment: LDS byte offset of this lane's row, and of the zeros its absent pieces read.
        struct FragmentRow
        {
            uint32_t offset; // of piece 0
            bool     live;
        };
        ROCWMMA_DEVICE inline FragmentRow fragmentRow(SampleShape const& s, uint32_t block, uint32_t lane)
        {
            const uint32_t row = block * 16u + (lane & 15u);
            return {row * s.pitch * 16u, row < s.m};
        }
        // 16 bytes of K of the lane's row: piece 4 step + lane / 16 (32 halves or 16 floats of K per step)
        ROCWMMA_DEVICE inline u32x4_t readRow(const char* tile, SampleShape const& s, FragmentRow const& r, uint32_t step, uint32_t lane)
        {
            const uint32_t piece = step * 4u + (lane >> 4);
            const uint32_t at    = r.live && piece < s.pieces ? r.offset + piece * 16u : s.m * s.pitch * 16u;
            return *reinterpret_cast<const u32x4_t*>(tile + at);
        }

        // acc(row of y, 4 columns of x) += one step; lane l holds row l % 16 of y's block, columns 4 (l / 16) .. + 3 of x's
        ROCWMMA_DEVICE inline f32x4_t multiplyStep(float16_t, u32x4_t x, u32x4_t y, f32x4_t acc)
        {
#if ROCWMMA_ARCH_GFX950
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, x), __builtin_bit_cast(f16x8_t, y), acc, 0, 0, 0);
#else
            (void)x, (void)y;
            return acc;
#endif
        }
        ROCWMMA_DEVICE inline f32x4_t multiplyStep(float32_t, u32x4_t x, u32x4_t y, f32x4_t acc)
        {
#if ROCWMMA_ARCH_GFX950
            const f32x4_t fx = __builtin_bit_cast(f32x4_t, x), fy = __builtin_bit_cast(f32x4_t, y);
#pragma unroll
            for(uint32_t t = 0; t < 4u; ++t)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fx[t], fy[t], acc, 0, 0, 0);
#else
            (void)x, (void)y;
#endif
            return acc;
        }

        // ------------------------------------------------------------------ forward
        // 16 bytes at an address aligned to its elements only (packed rows start anywhere)
        struct __attribute__((packed, aligned(2))) UnalignedPiece
        {
            uint32_t w[4];
        };
        ROCWMMA_DEVICE inline void storeUnaligned(void* to, u32x4_t v)
        {
            *static_cast<UnalignedPiece*>(to) = UnalignedPiece{{v[0], v[1], v[2], v[3]}};
        }

        // Slots: 16 x 16 blocks of the lower triangle per wave; block `part + PerSample * slot` in row-major order
        // (0,0), (1,0), (1,1), (2,0), ...  All of a wave's results stay in registers until every wave has read the
        // features, whose place the packed triangle then takes.
        template <typename T, uint32_t PerSample, uint32_t Slots>
        __global__ void __launch_bounds__(64 * wavesOf(PerSample)) dlrmFwdSampleKernel(const T* __restrict__ input, T* __restrict__ output, SampleShape s)
        {
            extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];
            const uint32_t lane   = threadIdx.x & 63u;
            const uint32_t wave   = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            const uint32_t part   = wave % PerSample; // this wave's part of its sample
            const uint32_t sample = blockIdx.x * (wavesOf(PerSample) / PerSample) + wave / PerSample;
            const bool     here   = sample < s.batch; // (wave uniform)
            char*          tile   = ldsRaw + (wave / PerSample) * s.sampleBytes;
            T* const       dst    = output + static_cast<size_t>(sample) * s.width;
            if(here)
                loadFeatures<PerSample>(tile, input + static_cast<size_t>(sample) * s.m * s.k, s, part, lane);
            lds::waitCopiesAndReads<0>();
            sampleSync<PerSample>();
            const uint32_t blocks = (s.m + 15u) / 16u, steps = (s.pieces + 3u) / 4u;
            f32x4_t        acc[Slots];
            uint32_t       rowOf[Slots], columnOf[Slots]; // (wave uniform)
            if(here)
            {
                // bottom-MLP row: the sample's first feature row
                for(uint32_t piece = part * 64u + lane; piece < s.pieces; piece += PerSample * 64u)
                    storeUnaligned(reinterpret_cast<char*>(dst) + piece * 16u, *reinterpret_cast<const u32x4_t*>(tile + piece * 16u));
                uint32_t I = 0u, J = part;
#pragma unroll
                for(uint32_t slot = 0; slot < Slots; ++slot)
                {
                    while(J > I)
                        J -= ++I;
                    rowOf[slot]    = I;
                    columnOf[slot] = J;
                    acc[slot]      = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    if(I < blocks)
                    {
                        const FragmentRow y = fragmentRow(s, I, lane), x = fragmentRow(s, J, lane);
#pragma unroll 4
                        for(uint32_t step = 0; step < steps; ++step)
                            acc[slot] = multiplyStep(T{}, readRow(tile, s, x, step, lane), readRow(tile, s, y, step, lane), acc[slot]);
                    }
                    J += PerSample;
                }
            }
            sampleSync<PerSample>();
            // the packed triangle, at an LDS address congruent to its global address modulo 16
            T* const       triangle = dst + s.k;
            T* const       out      = reinterpret_cast<T*>(tile + (reinterpret_cast<uintptr_t>(triangle) & 15u));
            const uint32_t entries  = s.width - s.k;
            if(here)
            {
#pragma unroll
                for(uint32_t slot = 0; slot < Slots; ++slot)
                    if(rowOf[slot] < blocks)
                    {
                        const uint32_t R     = rowOf[slot] * 16u + (lane & 15u);
                        const uint32_t start = (R * (R - 1u)) / 2u, C = columnOf[slot] * 16u + 4u * (lane >> 4);
                        // (entries outside the triangle go to a spare element behind it)
#pragma unroll
                        for(uint32_t e = 0; e < 4u; ++e)
                            out[R < s.m && C + e < R ? start + C + e : entries] = static_cast<T>(acc[slot][e]);
                    }
            }
            sampleSync<PerSample>();
            if(here)
            {
                constexpr uint32_t PerPiece = 16u / sizeof(T);
                const uint32_t     skew     = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(triangle) & 15u) / static_cast<uint32_t>(sizeof(T));
                const uint32_t     head     = min(entries, (PerPiece - skew) & (PerPiece - 1u));
                const uint32_t     whole    = (entries - head) / PerPiece, tail = head + whole * PerPiece;
                for(uint32_t i = part * 64u + lane; i < whole; i += PerSample * 64u)
                    reinterpret_cast<u32x4_t*>(triangle + head)[i] = reinterpret_cast<const u32x4_t*>(out + head)[i];
                if(part == 0u)
                {
                    if(lane < head)
                        triangle[lane] = out[lane];
                    if(tail + lane < entries)
                        triangle[tail + lane] = out[tail + lane];
                }
            }
        }

        // ------------------------------------------------------------------ backward
        // F operand: column n0 + lane % 16 of the contraction rows of one step (32 rows of halves, 16 of floats)
        ROCWMMA_DEVICE inline u32x4_t readColumns(float16_t, const char* tile, SampleShape const& s, uint32_t n0, uint32_t step, uint32_t lane)
        {
#if ROCWMMA_ARCH_GFX950
            u32x4_t x;
#pragma unroll
            for(uint32_t h = 0; h < 2u; ++h)
            {
                // a transposing read of four rows: the lane's 8 bytes of row 32 step + 8 (lane / 16) + 4 h + (lane % 16) / 4
                const uint32_t c  = step * 32u + (lane >> 4) * 8u + h * 4u + ((lane & 15u) >> 2);
                const uint32_t at = min(c, s.m) * s.pitch * 16u + n0 * 2u + ((lane & 3u) << 3);
                const auto     v  = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4_t*)(reinterpret_cast<uintptr_t>((lds::LdsPtr)(const_cast<char*>(tile) + at)))));
                x[2u * h]      = v[0];
                x[2u * h + 1u] = v[1];
            }
            return x;
#else
            (void)tile, (void)s, (void)n0, (void)step, (void)lane;
            return u32x4_t{};
#endif
        }
        ROCWMMA_DEVICE inline u32x4_t readColumns(float32_t, const char* tile, SampleShape const& s, uint32_t n0, uint32_t step, uint32_t lane)
        {
            u32x4_t x;
#pragma unroll
            for(uint32_t t = 0; t < 4u; ++t)
            {
                const uint32_t c = step * 16u + (lane >> 4) * 4u + t;
                x[t] = *reinterpret_cast<const uint32_t*>(tile + min(c, s.m) * s.pitch * 16u + (n0 + (lane & 15u)) * 4u);
            }
            return x;
        }

        // Stores two neighbouring 16-column blocks of a block row: 64 contiguous bytes per row and instruction.
        ROCWMMA_DEVICE inline void storeBlocks(float16_t* grad, SampleShape const& s, uint32_t row, uint32_t n0, f32x4_t a, f32x4_t b, uint32_t lane)
        {
            // the second block's run of a lane in an even 16-lane row changes places with the first block's of its
            // partner in the next one: every lane then owns eight consecutive columns
            uint32_t  x[2], y[2];
            float16_t h[4];
#pragma unroll
            for(uint32_t e = 0; e < 4u; ++e)
                h[e] = static_cast<float16_t>(a[e]);
            __builtin_memcpy(x, h, 8);
#pragma unroll
            for(uint32_t e = 0; e < 4u; ++e)
                h[e] = static_cast<float16_t>(b[e]);
            __builtin_memcpy(y, h, 8);
#if ROCWMMA_ARCH_GFX950
#pragma unroll
            for(uint32_t w = 0; w < 2u; ++w)
            {
                auto r = __builtin_amdgcn_permlane16_swap(x[w], y[w], false, false);
                x[w]   = r[0];
                y[w]   = r[1];
            }
#endif
            const uint32_t group = lane >> 4, column = n0 + (group & 1u) * 16u + 4u * (group & 2u);
            if(row < s.m && column < s.k)
                *reinterpret_cast<u32x4_t*>(grad + static_cast<size_t>(row) * s.k + column) = u32x4_t{x[0], x[1], y[0], y[1]};
        }
        ROCWMMA_DEVICE inline void storeBlocks(float32_t* grad, SampleShape const& s, uint32_t row, uint32_t n0, f32x4_t a, f32x4_t b, uint32_t lane)
        {
            const uint32_t column = n0 + 4u * (lane >> 4);
            if(row < s.m && column < s.k)
                *reinterpret_cast<u32x4_t*>(grad + static_cast<size_t>(row) * s.k + column) = __builtin_bit_cast(u32x4_t, a);
            if(row < s.m && column + 16u < s.k)
                *reinterpret_cast<u32x4_t*>(grad + static_cast<size_t>(row) * s.k + column + 16u) = __builtin_bit_cast(u32x4_t, b);
        }

        // G fragment: entries (R, c0 .. ) of the symmetric matrix with zero diagonal, from the packed triangle in LDS: below
        // the diagonal a row's entries are consecutive (tri(R) + c), above it entry (c, R) sits at tri(c) + R.  Every
        // entry is read (a harmless address where there is none) and selected afterwards, so the reads issue back to back.
        template <typename T>
        ROCWMMA_DEVICE inline u32x4_t readSymmetric(const T* triangle, uint32_t m, uint32_t R, uint32_t c0)
        {
            constexpr uint32_t N = 16u / sizeof(T);
            T                  v[N];
            uint32_t           above = (c0 * (c0 - 1u)) / 2u + R; // (c0 = 0: the product wraps to 0)
            const uint32_t     below = (R * (R - 1u)) / 2u;
#pragma unroll
            for(uint32_t j = 0; j < N; ++j)
            {
                const uint32_t c     = c0 + j;
                const bool     there = (c > R ? c : R) < m && c != R;
                const T        g     = triangle[there ? (c < R ? below + c : above) : 0u];
                v[j]                 = there ? g : static_cast<T>(0);
                above += c;
            }
            u32x4_t r;
            __builtin_memcpy(&r, v, 16);
            return r;
        }

        // MaxSteps: contraction steps the kernel is built for (the G fragments of a block row are held in registers)
        template <typename T, uint32_t PerSample, uint32_t MaxSteps>
        __global__ void __launch_bounds__(64 * wavesOf(PerSample)) dlrmBwdSampleKernel(const T* __restrict__ input, const T* __restrict__ upstream,
                                                                           T* __restrict__ grad, T* __restrict__ mlpGrad, SampleShape s)
        {
            extern __shared__ __attribute__((aligned(1024))) char ldsRaw[];
            constexpr uint32_t StepRows = 64u / sizeof(T); // contraction rows per step: 32 or 16
            constexpr uint32_t PerPiece = 16u / sizeof(T);
            const uint32_t     lane     = threadIdx.x & 63u;
            const uint32_t     wave     = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            const uint32_t     part     = wave % PerSample;
            const uint32_t     sample   = blockIdx.x * (wavesOf(PerSample) / PerSample) + wave / PerSample;
            const bool         here     = sample < s.batch; // (wave uniform)
            char*              tile     = ldsRaw + (wave / PerSample) * s.sampleBytes;
            char*              packed   = tile + s.featBytes;
            const uint32_t     steps    = (s.m + StepRows - 1u) / StepRows;
            // the upstream row starts on a boundary of its elements only: it is copied from the 4-byte boundary below it
            // (for halves possibly the previous sample's last entry) and read that much further on; an odd last half is
            // moved by hand, so nothing is read past the row's end
            const T*       up   = upstream + static_cast<size_t>(sample) * s.width;
            const uint32_t skew = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(up) & 3u); // 0 or 2 bytes
            if(here)
            {
                const char*           from  = reinterpret_cast<const char*>(up) - skew;
                const uint32_t        bytes = skew + s.width * static_cast<uint32_t>(sizeof(T)), words = bytes & ~3u;
                const lds::BufferRsrc rsrc  = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(from), 0, static_cast<int>(words), 0x00020000);
                for(uint32_t copy = part; copy * 1024u < words; copy += PerSample)
                    lds::asyncCopy16Streaming(packed + copy * 1024u, rsrc, copy * 1024u + lane * 16u, 0u);
                loadFeatures<PerSample>(tile, input + static_cast<size_t>(sample) * s.m * s.k, s, part, lane);
                lds::waitCopiesAndReads<0>();
                // (behind the copies, whose last lanes may have stored a zero there)
                if(words != bytes && (words / 1024u) % PerSample == part && lane == 0u)
                    *reinterpret_cast<uint16_t*>(packed + words) = *reinterpret_cast<const uint16_t*>(from + words);
            }
            sampleSync<PerSample>();
            if(here)
            {
                const T* row = reinterpret_cast<const T*>(packed + skew);
                // bottom-MLP gradient = the first k entries of the upstream row
                for(uint32_t piece = part * 64u + lane; piece < s.pieces; piece += PerSample * 64u)
                {
                    T v[PerPiece];
#pragma unroll
                    for(uint32_t e = 0; e < PerPiece; ++e)
                        v[e] = row[piece * PerPiece + e];
                    u32x4_t w;
                    __builtin_memcpy(&w, v, 16);
                    reinterpret_cast<u32x4_t*>(mlpGrad + static_cast<size_t>(sample) * s.k)[piece] = w;
                }
                T*             dst    = grad + static_cast<size_t>(sample) * s.m * s.k;
                const uint32_t blocks = (s.m + 15u) / 16u, pairs = (s.k + 31u) / 32u, units = blocks * pairs;
                u32x4_t        g[MaxSteps];
                uint32_t       heldBlock = ~0u;
                for(uint32_t u = units * part / PerSample; u < units * (part + 1u) / PerSample; ++u)
                {
                    const uint32_t I = u / pairs, n0 = (u - I * pairs) * 32u;
                    if(I != heldBlock) // (wave uniform)
                    {
                        heldBlock = I;
#pragma unroll
                        for(uint32_t step = 0; step < MaxSteps; ++step)
                            if(step < steps)
                                g[step] = readSymmetric(row + s.k, s.m, I * 16u + (lane & 15u), step * StepRows + PerPiece * (lane >> 4));
                    }
                    f32x4_t a = {0.0f, 0.0f, 0.0f, 0.0f}, b = a;
#pragma unroll
                    for(uint32_t step = 0; step < MaxSteps; ++step)
                        if(step < steps)
                        {
                            a = multiplyStep(T{}, readColumns(T{}, tile, s, n0, step, lane), g[step], a);
                            b = multiplyStep(T{}, readColumns(T{}, tile, s, n0 + 16u, step, lane), g[step], b);
                        }
                    storeBlocks(dst, s, I * 16u + (lane & 15u), n0, a, b, lane);
                }
            }
        }

        // ------------------------------------------------------------------ launch
        template <typename Kernel>
        int optInLds(Kernel kernel, uint32_t lds)
        {
            if(lds > 65536u
               && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds))
                      != hipSuccess)
                return ROCWMMA_AMD_LAUNCH_FAILED;
            return ROCWMMA_AMD_OK;
        }

        SampleShape shapeOf(uint32_t m, uint32_t k, uint32_t batch, uint32_t size, bool backward)
        {
            SampleShape s{};
            s.m          = m;
            s.k          = k;
            s.batch      = batch;
            s.pieces     = k * size / 16u;
            s.pitch      = s.pieces < 3u ? 3u : s.pieces | 1u; // (the division below needs more than one)
            s.pitchMagic = static_cast<uint32_t>((0x100000000ull + s.pitch - 1u) / s.pitch);
            // (a fragment of the last columns reads up to 64 bytes past its row)
            s.featBytes = ((m + 1u) * s.pitch * 16u + 64u + 1023u) & ~1023u;
            s.width     = k + m * (m - 1u) / 2u;
            // forward: the packed triangle takes the features' place (at its global address modulo 16, a spare element
            // behind it); backward: the upstream row behind the features
            const uint32_t packed = ((s.width + 1u) * size + 16u + 1023u) & ~1023u;
            s.sampleBytes         = backward ? s.featBytes + packed : (s.featBytes > packed ? s.featBytes : packed);
            return s;
        }

        // Waves per sample.  The LDS decides how many samples a compute unit works on at a time; the waves per sample make
        // those into enough waves to hide each other's loads and barriers (20 or more), and no more than that (every
        // wave of a sample waits for the slowest).  Measured with 1 / 2 / 4 / 8 waves, forward: 27 x 48 f16 (4 KiB)
        // 12.5 / 14.6 / 19.2 / 32.3 us, 45 x 128 f16 (13 KiB) 36.1 / 32.0 / 30.8 / 37.4, 94 x 232 f16 (44 KiB)
        // - / - / 65.0 / 56.1; backward: 41 x 72 f16 (6 KiB) 27.3 / 25.7 / 27.7 / 37.3, 123 x 24 f16 (15 KiB of triangle)
        // 143 / 73 / 69 / 76, 128 x 256 f16 (67 KiB) - / - / 105 / 82.  Both directions go by the same figure, so that a
        // sample is on the same XCD in both and backward finds its features in that L2 (27 x 128 f16, batch 2048,
        // forward + backward with 2 + 2 waves 13.2 us, with 1 + 2 14.1).  Small batches take more waves until the
        // device has 20 per compute unit (batch 1024, backward: 5.7 / 5.1 / 5.1 us).
        uint32_t wavesPerSample(SampleShape const& s, bool backward)
        {
            const uint32_t packed = s.width * (s.pieces * 16u / s.k), kib = (s.featBytes > packed ? s.featBytes : packed) / 1024u;
            uint32_t       per    = kib <= 5u ? 1u : kib <= 9u ? 2u : kib <= 30u ? 4u : 8u;
            while(per < 4u && static_cast<uint64_t>(s.batch) * per < 20u * computeUnits())
                per *= 2u;
            // forward: at most ten blocks of the triangle per wave
            const uint32_t blocks = ceilDiv(s.m, 16u), triangle = blocks * (blocks + 1u) / 2u;
            while(!backward && ceilDiv(triangle, per) > 10u)
                per *= 2u;
            while(s.sampleBytes * (wavesOf(per) / per) > kLdsBytes)
                per *= 2u;
            return per;
        }

        template <typename T, uint32_t PerSample, uint32_t Max>
        int launchFwd(const void* input, void* output, SampleShape const& s, hipStream_t stream)
        {
            auto           kernel = dlrmFwdSampleKernel<T, PerSample, Max>;
            const uint32_t lds    = s.sampleBytes * (wavesOf(PerSample) / PerSample);
            if(int rc = optInLds(kernel, lds))
                return rc;
            constexpr uint32_t perGroup = wavesOf(PerSample) / PerSample, threads = 64u * wavesOf(PerSample);
            return forEachLaunch(s.batch, threads, perGroup, [&](uint32_t first, uint32_t count) {
                SampleShape part = s;
                part.batch       = count;
                hipLaunchKernelGGL(kernel, dim3(ceilDiv(count, perGroup)), dim3(threads), lds, stream,
                                   static_cast<const T*>(input) + static_cast<size_t>(first) * s.m * s.k,
                                   static_cast<T*>(output) + static_cast<size_t>(first) * s.width, part);
                return launchStatus();
            });
        }
        template <typename T, uint32_t PerSample, uint32_t Max>
        int launchBwd(const void* input, const void* upstream, void* grad, void* mlpGrad, SampleShape const& s, hipStream_t stream)
        {
            auto           kernel = dlrmBwdSampleKernel<T, PerSample, Max>;
            const uint32_t lds    = s.sampleBytes * (wavesOf(PerSample) / PerSample);
            if(int rc = optInLds(kernel, lds))
                return rc;
            constexpr uint32_t perGroup = wavesOf(PerSample) / PerSample, threads = 64u * wavesOf(PerSample);
            return forEachLaunch(s.batch, threads, perGroup, [&](uint32_t first, uint32_t count) {
                SampleShape  part     = s;
                const size_t features = static_cast<size_t>(first) * s.m * s.k;
                part.batch            = count;
                hipLaunchKernelGGL(kernel, dim3(ceilDiv(count, perGroup)), dim3(threads), lds, stream, static_cast<const T*>(input) + features,
                                   static_cast<const T*>(upstream) + static_cast<size_t>(first) * s.width, static_cast<T*>(grad) + features,
                                   static_cast<T*>(mlpGrad) + static_cast<size_t>(first) * s.k, part);
                return launchStatus();
            });
        }

        template <typename T, uint32_t PerSample>
        int fwdByRows(const void* input, void* output, SampleShape const& s, hipStream_t stream)
        {
            const uint32_t blocks = ceilDiv(s.m, 16u), slots = ceilDiv(blocks * (blocks + 1u) / 2u, PerSample);
            if(slots <= 3u)
                return launchFwd<T, PerSample, 3>(input, output, s, stream);
            if(slots <= 6u)
                return launchFwd<T, PerSample, 6>(input, output, s, stream);
            return launchFwd<T, PerSample, 10>(input, output, s, stream); // (wavesPerSample: no more than ten)
        }
        template <typename T, uint32_t PerSample>
        int bwdByRows(const void* input, const void* upstream, void* grad, void* mlpGrad, SampleShape const& s, hipStream_t stream)
        {
            constexpr uint32_t Per32 = sizeof(T) == 2u ? 1u : 2u; // steps per 32 rows
            if(s.m <= 32u)
                return launchBwd<T, PerSample, Per32>(input, upstream, grad, mlpGrad, s, stream);
            if(s.m <= 64u)
                return launchBwd<T, PerSample, 2u * Per32>(input, upstream, grad, mlpGrad, s, stream);
            if(s.m <= 128u)
                return launchBwd<T, PerSample, 4u * Per32>(input, upstream, grad, mlpGrad, s, stream);
            return launchBwd<T, PerSample, 6u * Per32>(input, upstream, grad, mlpGrad, s, stream);
        }
    } // namespace

    int launchDlrmFwdSample(int dtype, const void* input, void* output, uint32_t m, uint32_t k, uint32_t batch, hipStream_t stream)
    {
        const uint32_t    size = dtype == ROCWMMA_AMD_F16 ? 2u : 4u;
        const SampleShape s    = shapeOf(m, k, batch, size, false);
        if(m > kMaxRows || s.sampleBytes > kLdsBytes)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        // The 128 x 128 tiles of a few large samples (three each from 129 rows on) run side by side where one workgroup per
        // sample leaves units idle: float32 180 x 160 batch 64 22.4 -> 17.4 us, 192 x 136 20.9 -> 17.5, but not up to 160 rows (160 x 200
        // 10.5 here) nor at narrow ones.  float16 samples of more than half the LDS have a unit to themselves: as tiles where those
        // fill the device better, 192 x 256 batch 64 11.1 -> 8.4, and from two samples per unit on, 192 x 256 batch 1024 56.9 -> 44.5, 96 x 512
        // 34.9 -> 26.3.
        const uint32_t units = computeUnits();
        const bool     fewTiles = m > 128u && 3u * static_cast<uint64_t>(batch) <= units;
        if(size == 4u ? fewTiles && m > 160u && k >= 64u : s.sampleBytes > kLdsBytes / 2u && (fewTiles || batch > units))
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t perSample = wavesPerSample(s, false);
        if(dtype == ROCWMMA_AMD_F16)
            return perSample == 1u   ? fwdByRows<float16_t, 1>(input, output, s, stream)
                   : perSample == 2u ? fwdByRows<float16_t, 2>(input, output, s, stream)
                   : perSample == 4u ? fwdByRows<float16_t, 4>(input, output, s, stream)
                                     : fwdByRows<float16_t, 8>(input, output, s, stream);
        return perSample == 1u   ? fwdByRows<float32_t, 1>(input, output, s, stream)
               : perSample == 2u ? fwdByRows<float32_t, 2>(input, output, s, stream)
               : perSample == 4u ? fwdByRows<float32_t, 4>(input, output, s, stream)
                                 : fwdByRows<float32_t, 8>(input, output, s, stream);
    }

    int launchDlrmBwdSample(int dtype, const void* input, const void* upstream, void* grad, void* mlpGrad, uint32_t m, uint32_t k,
                            uint32_t batch, hipStream_t stream)
    {
        const uint32_t    size = dtype == ROCWMMA_AMD_F16 ? 2u : 4u;
        const SampleShape s    = shapeOf(m, k, batch, size, true);
        if(m > kMaxRows || s.sampleBytes > kLdsBytes)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        // float32, wide samples in a batch that leaves units idle: 128-column tiles of their own (64 x 512 batch 64 15.9 -> 13.1 us,
        // 40 x 700 batch 16 12.3 -> 10.6)
        if(size == 4u && k > 256u && static_cast<uint64_t>(ceilDiv(k, 128u)) * batch <= computeUnits())
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t perSample = wavesPerSample(s, true);
        if(dtype == ROCWMMA_AMD_F16)
            return perSample == 1u   ? bwdByRows<float16_t, 1>(input, upstream, grad, mlpGrad, s, stream)
                   : perSample == 2u ? bwdByRows<float16_t, 2>(input, upstream, grad, mlpGrad, s, stream)
                   : perSample == 4u ? bwdByRows<float16_t, 4>(input, upstream, grad, mlpGrad, s, stream)
                                     : bwdByRows<float16_t, 8>(input, upstream, grad, mlpGrad, s, stream);
        return perSample == 1u   ? bwdByRows<float32_t, 1>(input, upstream, grad, mlpGrad, s, stream)
               : perSample == 2u ? bwdByRows<float32_t, 2>(input, upstream, grad, mlpGrad, s, stream)
               : perSample == 4u ? bwdByRows<float32_t, 4>(input, upstream, grad, mlpGrad, s, stream)
                                 : bwdByRows<float32_t, 8>(input, upstream, grad, mlpGrad, s, stream);
    }
} // namespace rocwmma_amd
