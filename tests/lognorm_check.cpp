// Host check of hm::half_log10 (henon_map_cpp_amd/csrc/hm_lognorm.h) against
// long double: the largest absolute error of log10(F)/2 beyond the rounding of
// the result, as a multiple of 2^-53 max(|result|, 2^-2), over log-uniform arguments of the
// normal and subnormal range, arguments in [0.5, 2] and both ends of every table
// bin; and the infinite and NaN arguments. Prints "max_error specials_ok".
#include <cmath>
#include <cstdio>
#include <random>

#include "hm_lognorm.h"

int main()
{
    hm::LogBin tab[hm::kLogBins];
    for (int i = 0; i < hm::kLogBins; ++i) tab[i] = hm::log_bin(i);
    std::mt19937_64 g(12345);
    std::uniform_real_distribution<double> e(-320.0, 308.0), a(0.5, 2.0);
    double worst = 0.0;
    auto check = [&](double x) {
        const long double want = 0.5L * log10l((long double)x);
        const double err = (double)fabsl((long double)hm::half_log10(x, tab) - want);
        worst = std::fmax(worst, err / (0x1p-53 * std::fmax(0.25, std::fabs((double)want))));
    };
    for (int i = 0; i < 2000000; ++i) check(std::pow(10.0, e(g)));
    for (int i = 0; i < 2000000; ++i) check(a(g));
    for (int k = -300; k <= 300; k += 7)
        for (int i = 0; i <= hm::kLogBins; ++i) {
            const double edge = std::ldexp(0.5 + i / (2.0 * hm::kLogBins), k);
            check(edge);
            check(std::nextafter(edge, 0.0));
        }
    const bool ok = hm::half_log10(INFINITY, tab) == INFINITY && std::isnan(hm::half_log10(NAN, tab));
    std::printf("%.3f %d\n", worst, ok ? 1 : 0);
    return 0;
}
