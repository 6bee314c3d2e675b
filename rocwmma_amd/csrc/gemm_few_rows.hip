// GEMM for few token rows: element types and the choice against the blocked kernel.  The kernel is in gemm_few_rows.hpp.
#include "gemm_few_rows.hpp"
#include "gemm_blocked_rungs.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmFewRows(int dtypeIn, int dtypeOut, int layoutA, int layoutB, GemmArgs& g, hipStream_t stream)
    {
        if(dtypeIn == ROCWMMA_AMD_F32)
            return ROCWMMA_AMD_UNSUPPORTED_TYPE;
        if(layoutA != ROCWMMA_AMD_ROW_MAJOR || layoutB != ROCWMMA_AMD_COL_MAJOR || g.layoutC != ROCWMMA_AMD_ROW_MAJOR
           || g.m % 16u != 0u || g.n % 16u != 0u)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const bool        half   = dtypeIn == ROCWMMA_AMD_F16 || dtypeIn == ROCWMMA_AMD_BF16;
        const OperandKind kind   = half ? OperandKind::Half : (dtypeIn == ROCWMMA_AMD_I8 ? OperandKind::Int8 : OperandKind::Fp8);
        const uint64_t    kBytes = static_cast<uint64_t>(g.k) * (half ? 2u : 1u);
        const uint32_t    outBytes = dtypeOut == ROCWMMA_AMD_F32 || dtypeOut == ROCWMMA_AMD_I32 ? 4u : (dtypeOut == ROCWMMA_AMD_I8 ? 1u : 2u);
        if(kBytes <= kFewStep) // (as cheapestFew has it, without the call that asks for the units)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        const uint32_t  units   = computeUnits();
        const FewChoice few     = cheapestFew(g.m, g.n, kBytes, units);
        float           blocked = 0.0f;
        if(few.mb == 0u)
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        // (handed on: estimating all rungs takes 50 to 100 ns, which a small call notices, and the blocked kernel would do it again)
        const Rung rung = cheapestRung(kind, layoutPair(true, true), g.m, g.n, kBytes, outBytes, units, waveTileTakes(g), &blocked);
        if(few.time * kFewMargin > blocked)
        {
            g.rung = static_cast<uint8_t>(rung);
            return ROCWMMA_AMD_UNSUPPORTED_SHAPE;
        }
        if(dtypeIn == ROCWMMA_AMD_F16 && dtypeOut == ROCWMMA_AMD_F32)
            return launchFewRows<float16_t, float32_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_F16 && dtypeOut == ROCWMMA_AMD_F16)
            return launchFewRows<float16_t, float16_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_BF16 && dtypeOut == ROCWMMA_AMD_F32)
            return launchFewRows<bfloat16_t, float32_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_BF16 && dtypeOut == ROCWMMA_AMD_BF16)
            return launchFewRows<bfloat16_t, bfloat16_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_E4M3 && dtypeOut == ROCWMMA_AMD_F32)
            return launchFewRows<float8_t, float32_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_E5M2 && dtypeOut == ROCWMMA_AMD_F32)
            return launchFewRows<bfloat8_t, float32_t, float32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_I8 && dtypeOut == ROCWMMA_AMD_I32)
            return launchFewRows<int8_t, int32_t, int32_t>(g, stream, few);
        if(dtypeIn == ROCWMMA_AMD_I8 && dtypeOut == ROCWMMA_AMD_I8)
            return launchFewRows<int8_t, int8_t, int32_t>(g, stream, few);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

} // namespace rocwmma_amd
