// Host check of gd_sixth (godunov_kernels.h) against the division: the same bits
// for normal and subnormal numbers, zeros of both signs and infinities, NaN for NaN.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>

#include "godunov_kernels.h"

static uint64_t bits(double v) {
    uint64_t b;
    std::memcpy(&b, &v, 8);
    return b;
}

int main() {
    long bad = 0;
    auto check = [&](double x) {
        const double a = mgx::gd_sixth(x), b = x / 6.0;
        if (std::isnan(x) ? std::isnan(a) : bits(a) == bits(b)) return;
        if (bad++ < 10) std::printf("x %a: %a instead of %a\n", x, a, b);
    };
    const double inf = std::numeric_limits<double>::infinity(), big = std::numeric_limits<double>::max();
    for (double x : {0.0, inf, std::nan(""), big, 0x1p-960, 0x1p-1022}) {
        check(x);
        check(-x);
        check(std::nextafter(x, 0.0));
        check(-std::nextafter(x, inf));
    }
    for (int n = 1; n < 4000; ++n) check(n * 0x1p-1074);
    uint64_t s = 88172645463325252ull;  // xorshift64 (Marsaglia 2003)
    for (int e = 0; e < 2047; ++e)
        for (int t = 0; t < 2000; ++t) {
            s ^= s << 13;
            s ^= s >> 7;
            s ^= s << 17;
            const uint64_t b = (s & 0x800fffffffffffffull) | ((uint64_t)e << 52);
            double x;
            std::memcpy(&x, &b, 8);
            check(x);
        }
    std::printf("%ld differ\n", bad);
    return bad != 0;
}
