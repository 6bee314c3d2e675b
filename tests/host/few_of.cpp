// Reads problems (operand kind 0 half / 1 int8 / 2 fp8, m, n, bytes of K, bytes per element of D) and prints how many blocks of 16
// weight rows a workgroup of the kernel for few rows takes on 256 compute units, or 0 where the blocked kernel has the problem.
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
        std::printf("%u\n", few.time * kFewMargin > blocked ? 0u : few.nb);
    }
    return 0;
}
