// Counts quotients of divide() that are not the IEEE quotient: random and
// nearly-halfway numerators over the kinds of divisors the kernels use.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include "../../loki-mc_amd/csrc/common.h"
using namespace ekmc;

int main() {
    std::mt19937_64 rng(20240611);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    const double lo[] = {1e5, 1e-5, 1e18, 1e6, 1e-3}, hi[] = {1e14, 10.0, 1e27, 1e12, 1e3};
    long bad = 0, n = 0;
    auto check = [&](double x, double d, const Reciprocal& r) {
        const double a = divide(x, d, r), b = x / d;
        ++n;
        if (std::memcmp(&a, &b, 8) != 0 && !(a == 0 && b == 0)) ++bad;
    };
    for (int k = 0; k < 6; ++k)
        for (int j = 0; j < 2000; ++j) {
            const double d = k == 5 ? kCharge : lo[k] * std::pow(hi[k] / lo[k], u(rng));
            const Reciprocal r = k == 5 ? kChargeInv : reciprocal(d);
            if (k == 5 && (r.hi != reciprocal(d).hi || std::fabs(r.lo - reciprocal(d).lo) > 1e-10 * std::fabs(r.lo))) ++bad;
            check(0.0, d, r);
            for (int i = 0; i < 120; ++i) {
                const double x = (u(rng) - 0.3) * std::pow(10.0, 60.0 * u(rng) - 40.0);
                check(x, d, r);
                // numerators whose quotient lies next to a double or halfway between two
                const double q = x / d, up = std::nextafter(q, INFINITY);
                check(q * d, d, r);
                check((q * 0.5 + up * 0.5) * d, d, r);
                check(std::nextafter(q * d, 0.0), d, r);
                check(std::nextafter(q * d, INFINITY), d, r);
            }
        }
    std::printf("%ld %ld\n", bad, n);
    return bad != 0;
}
