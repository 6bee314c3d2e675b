// Reads problems (operand kind 0 half / 1 int8 / 2 fp8, m, n, bytes of K, bytes per element of D) and prints the tile
// (blocks of 16 rows of A, of 16 weight rows) of the kernel whose waves share K on 256 compute units, or 0 0 where the blocked kernel
// has the problem.
#include "../../rocwmma_amd/csrc/gemm_blocked_rungs.hpp"
#include "../../rocwmma_amd/csrc/gemm_few_rows_rule.hpp"

#include <cstdio>

using namespace rocwmma_amd;

int main()
{
    unsigned           kind, m, n, out;
    unsigned long long kBytes;
    while(std::scanf("%u %u %u %llu %u", &kind, &m, &n, &kBytes, &out) == 5)
    {
        float blocked = 0.0f;
        cheapestRung(static_cast<OperandKind>(kind), 0u, m, n, kBytes, out, 256u, true, &blocked);
        const FewChoice few = cheapestFew(m, n, kBytes, 256u);
        if(few.mb == 0u || few.time * kFewMargin > blocked)
            std::printf("0 0\n");
        else
            std::printf("%u %u\n", few.mb, few.nb);
    }
    return 0;
}
