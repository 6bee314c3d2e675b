// The blocked GEMM with bias and activation in its epilogue, f16 operands.
#include "gemm_blocked_ladder.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmFusedF16(int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream)
    {
        if(dtypeOut == ROCWMMA_AMD_F32)
            return pickLayout<float16_t, float32_t, float32_t, true>(layoutA, layoutB, g, stream, TileUse::Any);
        if(dtypeOut == ROCWMMA_AMD_F16)
            return pickLayout<float16_t, float16_t, float32_t, true>(layoutA, layoutB, g, stream, TileUse::Any);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

} // namespace rocwmma_amd
