// The blocked GEMM's tile ladder for int8 operands.
#include "gemm_blocked_ladder.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmBlockedI8(int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream, TileUse use)
    {
        if(dtypeOut == ROCWMMA_AMD_I32)
            return pickLayout<int8_t, int32_t, int32_t, false>(layoutA, layoutB, g, stream, use);
        if(dtypeOut == ROCWMMA_AMD_I8)
            return pickLayout<int8_t, int8_t, int32_t, false>(layoutA, layoutB, g, stream, use);
        return ROCWMMA_AMD_UNSUPPORTED_TYPE;
    }

} // namespace rocwmma_amd
