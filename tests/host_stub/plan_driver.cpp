// Prints what the size rules of the one-launch dispatch say about worlds (mooncake_amd/csrc/ep_plan.cpp compiled on the
// CPU).  A line of input is
//   <experts> <K> <hidden> <use_fp8> <fused_small_max> <fused_shared_max> <R> <tokens of rank 0> ... <tokens of rank R-1>
// and gives "<one launch: 0 or 1> <every wave by itself: 0 or 1> <tokens of a block>".
#include <cstdio>
#include <iostream>
#include <vector>

#include "ep_kernels.h"

int main() {
    int E, K, hidden, fp8, R;
    mcep::Tuning t;
    while (std::cin >> E >> K >> hidden >> fp8 >> t.fused_small_max >> t.fused_shared_max >> R) {
        std::vector<int32_t> n(R);
        for (auto& v : n) std::cin >> v;
        const mcep::SmallPlan p = mcep::plan_small(n.data(), R, E, K, hidden, fp8 != 0, t);
        std::printf("%d %d %d\n", (int)p.fused, (int)p.alone, p.block_tokens);
    }
    return 0;
}
