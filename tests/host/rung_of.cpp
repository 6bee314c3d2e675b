// Reads problems (operand kind 0 half / 1 int8 / 2 fp8, layout pair 0..3, m, n, bytes of K, bytes per element of D) and prints the
// rung the blocked GEMM runs each on, on 256 compute units; "rungs" prints every rung there is, per kind and layout pair.
#include "../../rocwmma_amd/csrc/gemm_blocked_rungs.hpp"

#include <cstdio>
#include <cstring>

using namespace rocwmma_amd;

static const char* const kNames[] = {"None", "Big", "Wide", "Mid", "MidLines", "Ring2", "Ring4", "NarrowLines", "Narrow", "Narrow64", "Tiny", "Tiny64", "WaveTile"};

int main(int argc, char** argv)
{
    if(argc > 1 && std::strcmp(argv[1], "rungs") == 0)
    {
        for(uint32_t kind = 0; kind < 3u; ++kind)
            for(uint32_t pair = 0; pair < 4u; ++pair)
                for(RungCost const& c : kRungTables[kind][pair].rungs)
                    if(c.rung != Rung::None)
                        std::printf("%u %u %s\n", kind, pair, kNames[static_cast<uint32_t>(c.rung)]);
        return 0;
    }
    unsigned           kind, pair, m, n, out;
    unsigned long long kBytes;
    while(std::scanf("%u %u %u %u %llu %u", &kind, &pair, &m, &n, &kBytes, &out) == 6)
        std::printf("%s\n", kNames[static_cast<uint32_t>(cheapestRung(static_cast<OperandKind>(kind), pair, m, n, kBytes, out, 256u, true))]);
    return 0;
}
