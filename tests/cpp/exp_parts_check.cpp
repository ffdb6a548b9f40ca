// Host build of the volumetric spectrum's exponentials (sirius_amd/csrc/geodesic.hpp) against FP64:
// expm1_pos on [1e-12, 88] and exp_neg on [-87, 0] within 4 units of 2^-24 (two roundings of the
// argument's reduction, of the polynomial and of the last sum), at the ends of each binade's
// reduction (multiples of ln(2) / 2) too, and held flat beyond 88. Prints the worst and "OK".
#include "../../sirius_amd/csrc/geodesic.hpp"

#include <cmath>
#include <cstdio>

using namespace sirius;

int main() {
    const double u = std::ldexp(1.0, -24);
    double worst1 = 0, worst2 = 0;
    auto check = [&](float x) {
        const double a = expm1_pos(x), b = std::expm1((double)x);
        worst1 = std::fmax(worst1, std::fabs(a - b) / (u * b));
        if (x <= 87.f) {
            const double c = exp_neg(-x), d = std::exp(-(double)x);
            worst2 = std::fmax(worst2, std::fabs(c - d) / (u * d));
        }
    };
    for (double x = 1e-12; x <= 88.0; x *= 1.00013) check((float)x);
    for (int k = 1; k < 254; ++k) {
        const float x = (float)(k * 0.34657359027997264);
        if (x >= 87.9f) break;
        check(x);
        check(std::nextafterf(x, 0.f));
        check(std::nextafterf(x, 100.f));
    }
    check(88.f);
    std::printf("expm1 %.2f exp %.2f units of 2^-24\n", worst1, worst2);
    const bool ends = expm1_pos(0.f) == 0.f && exp_neg(0.f) == 1.f && expm1_pos(1e30f) == expm1_pos(88.f) &&
                      expm1_pos(INFINITY) == expm1_pos(88.f) && exp_neg(-INFINITY) < 1e-37f && std::isfinite(expm1_pos(88.f));
    if (worst1 <= 4 && worst2 <= 4 && ends) std::puts("OK");
    return 0;
}
