// plan_launch (csrc/rt_common.hpp) at and around every line it draws.  Prints
// the number of plans looked at, then one line for each that breaks a rule.
#include <cstdio>
#include <vector>

#include "rt_common.hpp"

using rtamd::LaunchPlan;
using rtamd::plan_launch;

int main() {
    unsigned long long plans = 0;
    for (uint32_t cus : {1u, 4u, 32u, 255u, 256u, 304u}) {
        const uint32_t simds = cus * 4u;
        std::vector<uint64_t> ns = {1, 2, 3, 7, 8, 9, 63, 64, 65, 255, 256, 257, 1u << 22, 0x7fffffffu};
        for (uint64_t load : {1u, 8u, 9u, 64u, 128u, 192u, 193u, 256u, 320u, 321u, 447u, 448u, 449u, 1000u, 4096u})
            for (int d : {-1, 0, 1}) ns.push_back(load * simds + d);
        for (uint64_t n64 : ns) {
            if (n64 < 1 || n64 > 0x7fffffffu) continue;
            const uint32_t n = (uint32_t)n64;
            for (uint32_t waves : {2u, 4u})
                for (uint32_t per_cu = 1; per_cu <= 16u / waves * 2u; ++per_cu) {
                    const uint32_t grid = cus * per_cu;
                    const LaunchPlan p = plan_launch(n, grid, waves, simds);
                    const uint64_t w = (uint64_t)p.blocks * waves;
                    // a kernel plans again from its own grid: the same, or it would hand out other rays
                    const LaunchPlan q = plan_launch(n, p.blocks, waves, simds);
                    const bool ok = p.blocks >= 1 && p.blocks <= grid && p.per_wave <= 64 &&
                                    (p.per_wave ? p.per_wave * w >= n && (p.per_wave - 1) * w < n : n > 64 * w) &&
                                    q.blocks == p.blocks && q.per_wave == p.per_wave;
                    ++plans;
                    if (!ok)
                        std::printf("n %u cus %u waves %u grid %u: blocks %u per_wave %u, again %u %u\n", n, cus, waves,
                                    grid, p.blocks, p.per_wave, q.blocks, q.per_wave);
                }
        }
    }
    std::printf("%llu\n", plans);
    return 0;
}
