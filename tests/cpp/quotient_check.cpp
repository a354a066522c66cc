// quotient (csrc/rt_common.hpp) against the division, bit for bit: origins and
// scales of binary32, as a ray's setup has them.  Prints how many pairs were
// compared and how many differed.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "rt_common.hpp"

int main() {
    std::mt19937_64 rng(7);
    auto real = [&](int lo, int hi) {
        const double m = 1.0 + std::ldexp((double)(rng() >> 12), -52);
        const float f = (float)std::ldexp(m, lo + (int)(rng() % (uint64_t)(hi - lo)));
        return rng() & 1 ? -f : f;
    };
    unsigned long long pairs = 0, differ = 0;
    for (int k = 0; k < 4000000; ++k) {
        const float scale = std::fabs(k & 1 ? real(-24, -8) : real(-126, 100));
        const double x = k & 2 ? (double)real(-10, 10) - (double)real(-10, 10)
                               : (double)real(-126, 120) - (double)real(-126, 120);
        const double want = x / (double)scale, got = rtamd::quotient(x, (double)scale, 1.0 / (double)scale);
        differ += std::memcmp(&want, &got, 8) != 0;
        ++pairs;
    }
    std::printf("%llu %llu\n", pairs, differ);
    return 0;
}
