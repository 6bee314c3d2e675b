// The blocked GEMM's tile ladder for bf16 operands.
#include "gemm_blocked_ladder.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmBlockedBf16(int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream, TileUse use)
    {
        if(dtypeOut == ROCWMMA_AMD_F32)
            return pickLayout<bfloat16_t, float32_t, float32_t, false>(layoutA, layoutB, g, stream, use);
        if(dtypeOut == ROCWMMA_AMD_BF16)
            return pickLayout<bfloat16_t, bfloat16_t, float32_t, false>(layoutA, layoutB, g, stream, use);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

} // namespace rocwmma_amd
