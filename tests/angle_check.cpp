// Host check of hm::angle_of (henon_map_cpp_amd/csrc/hm_angle.h) against long
// double atan2: the largest error as a multiple of 2^-53 max(|result|, 2^-1000) over
// random points of all octants, points near the axes, the diagonals and the table's
// bin edges, magnitudes from subnormal to huge; and every pair of special values
// against std::atan2, signs of zeros included. Prints "max_error specials_ok".
#include <cmath>
#include <cstdio>
#include <random>

#include "hm_angle.h"

int main()
{
    std::mt19937_64 g(12345);
    std::uniform_real_distribution<double> a(-1.0, 1.0), e(-300.0, 300.0);
    double worst = 0.0;
    auto check = [&](double y, double x) {
        const long double want = atan2l((long double)y, (long double)x);
        if (fabsl(want) < 0x1p-1000L) return;
        const double err = (double)fabsl((long double)hm::angle_of(y, x, hm::kAtan) - want);
        worst = std::fmax(worst, err / (0x1p-53 * std::fabs((double)want)));
    };
    for (int k = 0; k < 3000000; ++k) check(a(g), a(g));
    for (int k = 0; k < 1000000; ++k) check(a(g) * std::pow(2.0, a(g) * 40), a(g));
    for (int k = 0; k < 1000000; ++k) {
        const double s = std::pow(10.0, e(g));
        check(a(g) * s, a(g) * s);
    }
    for (int k = 0; k < 1000000; ++k) {
        const double x = a(g);
        check(x * (1.0 + std::ldexp(a(g), -(k % 53))), k % 2 ? x : -x);
    }
    for (int i = 0; i <= 128; ++i)
        for (int k = 0; k < 200; ++k) {
            const double x = a(g), y = x * (i / 128.0);
            check(y, x);
            check(x, y);
            check(std::nextafter(y, 2.0), x);
            check(std::nextafter(y, -2.0), -x);
        }
    for (int k = 0; k < 1000; ++k) check(std::ldexp(a(g), -1050), std::ldexp(a(g), -1040));
    const double sp[] = {0.0, -0.0, 1.0, -1.0, 1e300, -1e300, 5e-324, -5e-324, INFINITY, -INFINITY, NAN, 1e-200, 0.5};
    int ok = 1;
    for (double y : sp)
        for (double x : sp) {
            const double gv = hm::angle_of(y, x, hm::kAtan), wv = std::atan2(y, x);
            if (std::isnan(wv) ? !std::isnan(gv)
                               : !(std::fabs(gv - wv) <= 4 * 0x1p-53 * std::fabs(wv) && std::signbit(gv) == std::signbit(wv)))
                ok = 0;
        }
    std::printf("%.3f %d\n", worst, ok);
    return 0;
}
