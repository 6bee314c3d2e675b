// Reads problems (operand kind 0 half / 1 int8 / 2 fp8, layout pair 0..3, m, n, bytes of K, bytes per element of D) and prints what
// rocwmma_amd_gemm runs each on, on 256 compute units with C and D row-major: a rung of the blocked GEMM, "Few" (the kernel whose waves
// share K), "Skinny" and the K steps that the weight-streaming kernel fetches together, or "Sliced".
#include "../../rocwmma_amd/csrc/gemm_blocked_rungs.hpp"
#include "../../rocwmma_amd/csrc/gemm_few_rows_rule.hpp"
#include "../../rocwmma_amd/csrc/gemm_skinny_rule.hpp"

#include <cstdio>

using namespace rocwmma_amd;

static const char* const kNames[] = {"None", "Big", "Wide", "Mid", "MidLines", "Ring2", "Ring4", "NarrowLines", "Narrow", "Narrow64", "Tiny", "Tiny64", "WaveTile"};

int main()
{
    unsigned           kind, pair, m, n, out;
    unsigned long long kBytes;
    while(std::scanf("%u %u %u %u %llu %u", &kind, &pair, &m, &n, &kBytes, &out) == 6)
    {
        float      blocked = 0.0f;
        const Rung rung    = cheapestRung(static_cast<OperandKind>(kind), pair, m, n, kBytes, out, 256u, true, &blocked);
        if(pair == 0u)
        {
            const uint32_t  steps = out == 4u ? skinnySteps(m, n, kBytes, 256u) : 0u;
            const FewChoice few   = cheapestFew(m, n, kBytes, 256u);
            if(steps != 0u || (out == 4u && kSlicesOf(m, n, kBytes, 256u) != 0u))
            {
                steps != 0u ? std::printf("Skinny%u\n", steps) : std::printf("Sliced\n");
                continue;
            }
            if(few.mb != 0u && few.time * kFewMargin <= blocked)
            {
                std::printf("Few\n");
                continue;
            }
        }
        std::printf("%s\n", kNames[static_cast<uint32_t>(rung)]);
    }
    return 0;
}
