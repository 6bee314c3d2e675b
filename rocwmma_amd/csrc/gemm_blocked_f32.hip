// The blocked GEMM's tiles for float32 operands.
#include "gemm_blocked_ladder.hpp"

using namespace rocwmma;

namespace rocwmma_amd
{
    int launchGemmBlockedF32(int dtypeOut, int layoutA, int layoutB, GemmArgs const& g, hipStream_t stream)
    {
        if(dtypeOut != ROCWMMA_AMD_F32)
            return ROCWMMA_AMD_UNSUPPORTED_TYPE;
        const bool ak = layoutA == ROCWMMA_AMD_ROW_MAJOR, bk = layoutB == ROCWMMA_AMD_COL_MAJOR;
        if(ak)
            return bk ? pickTileF32<true, true>(g, stream) : pickTileF32<true, false>(g, stream);
        return bk ? pickTileF32<false, true>(g, stream) : pickTileF32<false, false>(g, stream);
    }

} // namespace rocwmma_amd
