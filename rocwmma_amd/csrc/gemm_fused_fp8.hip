// The blocked GEMM with bias and activation in its epilogue, fp8 operands.
#include "gemm_blocked_ladder.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmFusedFp8(int dtypeIn, int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream)
    {
        if(dtypeIn == ROCWMMA_AMD_E4M3 && dtypeOut == ROCWMMA_AMD_F32)
            return pickLayout<float8_t, float32_t, float32_t, true>(layoutA, layoutB, g, stream, TileUse::Any);
        if(dtypeIn == ROCWMMA_AMD_E5M2 && dtypeOut == ROCWMMA_AMD_F32)
            return pickLayout<bfloat8_t, float32_t, float32_t, true>(layoutA, layoutB, g, stream, TileUse::Any);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

} // namespace rocwmma_amd
