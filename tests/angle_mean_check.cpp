// Host check of hm::angle_of (henon_map_cpp_amd/csrc/hm_angle.h): its mean error and that
// of the C library's atan2 against long double, in units of 2^-53 of the result, over
// points of all octants; and its largest error where the result is 1/64 at least.
// Prints "mean library_mean worst".
#include <cmath>
#include <cstdio>
#include <random>

#include "hm_angle.h"

int main()
{
    std::mt19937_64 g(54321);
    std::uniform_real_distribution<double> a(-1.0, 1.0);
    double sum = 0.0, lib = 0.0, worst = 0.0;
    const int n = 4000000;
    for (int k = 0; k < n; ++k) {
        const double y = a(g), x = a(g);
        const long double want = atan2l((long double)y, (long double)x);
        const double unit = 0x1p-53 * std::fabs((double)want);
        const double e = (double)fabsl((long double)hm::angle_of(y, x, hm::kAtan) - want) / unit;
        sum += e;
        lib += (double)fabsl((long double)std::atan2(y, x) - want) / unit;
        if (fabsl(want) >= 0x1p-6L) worst = std::fmax(worst, e);
    }
    std::printf("%.5f %.5f %.4f\n", sum / n, lib / n, worst);
    return 0;
}
