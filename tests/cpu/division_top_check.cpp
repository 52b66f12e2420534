// division_top_check.cpp -- the CH column solve's divisions for numerators from
// 2^900 to the largest finite one (no test of the kernel keeps them away): a
// finite result has to be the IEEE quotient; one that is not finite sends the
// step to IEEE division.  And the rule that lets the step's last value show it:
// what is not finite stays so through a row, whatever its factors.
//
// usage: division_top_check <samples> <seed>
// prints "<five-operation quotients> <finite> <wrong>", the same for the
// two-operation ones, and "<rows> <finite again>"
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#include "../../custen_amd/csrc/ch_setup.h"

namespace {

uint64_t state;
uint64_t next()  // SplitMix64
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// random sign and significand, exponent in [lo, hi]
double draw(int lo, int hi)
{
    const uint64_t r = next();
    const int e = lo + (int)(next() % (uint64_t)(hi - lo + 1));
    const double v = std::ldexp(1.0 + (double)(r >> 12) * 0x1p-52, e);
    return (r & 1) ? -v : v;
}

// numerators: any of the range, and those whose quotient by d lies at the top
double numerator(double d, int k)
{
    if (k % 3 == 0) return draw(900, 1023);
    const double q = std::ldexp(2.0 - (double)(next() % 64) * 0x1p-52, 1022);  // up to the largest
    const double n = q * d * (k % 3 == 1 ? 1.0 : 2.0);
    return std::isfinite(n) && std::fabs(n) >= 0x1p900 ? n : draw(1000, 1023);
}

struct Count {
    long tried = 0, finite = 0, wrong = 0;
    void add(double q, double ref)
    {
        tried++;
        if (!std::isfinite(q)) return;
        finite++;
        wrong += std::memcmp(&q, &ref, sizeof q) != 0;
    }
};

}  // namespace

int main(int argc, char** argv)
{
    if (argc != 3) return 2;
    const long samples = std::atol(argv[1]);
    state = std::strtoull(argv[2], nullptr, 10);
    Count five, two;
    while (five.tried < samples) {
        const double d = draw(-60, 59), n = numerator(d, (int)five.tried), y = 1.0 / d;
        double q = n * y;
        q = std::fma(std::fma(-d, q, n), y, q);
        five.add(std::fma(std::fma(-d, q, n), y, q), n / d);
    }
    while (two.tried < samples) {
        const double d = draw(-60, 59);
        if (!custen::chDivCertified(d)) continue;
        const double zh = 1.0 / d, zl = std::fma(-d, zh, 1.0) / d;
        for (int i = 0; i < 1000; i++) {
            const double n = numerator(d, i);
            two.add(std::fma(n, zh, n * zl), n / d);
        }
    }
    long rows = 0, finite = 0;
    const double factors[] = {0.0, -0.0, 5e-324, 1e-300, 1.0, -3.0, 1e300, DBL_MAX};
    for (double b1 : {(double)INFINITY, -(double)INFINITY, (double)NAN})
        for (double f1 : factors)
            for (double f0 : factors)
                for (double b2 : {0.0, 1.0, -1e308, (double)INFINITY, -(double)INFINITY})
                    for (double c : {0.0, -0.0, 1.0, -1e308, (double)INFINITY, (double)NAN}) {
                        const double num = (c - f0 * b2) - f1 * b1;
                        rows++;
                        finite += std::isfinite(num);
                    }
    std::printf("%ld %ld %ld\n%ld %ld %ld\n%ld %ld\n", five.tried, five.finite, five.wrong,
                two.tried, two.finite, two.wrong, rows, finite);
    return 0;
}
