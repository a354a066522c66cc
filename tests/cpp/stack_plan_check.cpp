// Prints plan_stack (csrc/rt_common.hpp) for every stack a launch may need:
// need, stack_lds asked for, crowded, then entries in LDS and whether the rest spill.
#include <cstdio>

#include "rt_common.hpp"

int main() {
    for (uint32_t need = 1; need <= rtamd::kMaxWideStack; ++need)
        for (uint32_t asked : {0u, 8u, 16u, 32u})
            for (bool crowded : {false, true}) {
                const rtamd::StackPlan p = rtamd::plan_stack(need, asked, crowded);
                std::printf("%u %u %d %u %d\n", need, asked, crowded, p.lds, p.deep);
            }
    return 0;
}
