// log10 of the tangent matrix's norm for the per-turn MEGNO sums: half_log10(F) =
// log10(sqrt(F)) for F = |M|_F^2, from a 256-entry table in LDS. F = 2^e m with m
// in [1/2, 1); the top eight mantissa bits choose c (1 / the bin's centre, rounded)
// and log10(1/c) / 2; with r = m c - 1 (one fused operation, |r| <= 2^-9)
//   log10(F) / 2 = e log10(2) / 2 + log10(1/c) / 2 + log10(1 + r) / 2,
// the last by five terms of its series (the sixth is below 2e-18).
// The MEGNO recursion needs log10(|M_{k+1}| / |M_k|) only: the difference of two
// consecutive values, each formed once, exponents and mantissas apart (log_ratio).
// Taking logarithms of norms instead of ratios drops the division (12 instructions on
// gfx950) and needs absolute, not relative, accuracy, so 12 instructions do for the
// logarithm where one accurate around 1 takes about 45. The rounding of one value
// enters the first MEGNO sum with weight k and leaves it with weight k + 1, so its net
// weight is 1, where the rounding of a ratio counts k times.
// Zero is the caller's case (the table gives a finite value); infinite and NaN
// arguments give themselves; subnormal ones are handled.
// Compiles as host code too (no HIP types), so a host check can build it alone.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#define HM_LOGNORM_FN __host__ __device__ inline
#else
#define HM_LOGNORM_FN inline
#endif

namespace hm {

constexpr int kLogBins = 256;
struct alignas(16) LogBin {
    double c, l;  // c = 1 / centre, l = log10(1/c) / 2
};

HM_LOGNORM_FN LogBin log_bin(int i)
{
    const double c = 1.0 / (0.5 + ((double)i + 0.5) / (2.0 * kLogBins));
    return LogBin{c, -0.5 * log10(c)};
}

constexpr double kHalfLog10Of2 = 0.15051499783199060;

// log10(sqrt(F)) = f + e log10(2) / 2, f in (-0.151, 0].
struct LogNorm {
    double f;
    int e;
};

HM_LOGNORM_FN LogNorm log_norm(double F, const LogBin *tab)
{
    constexpr double H = 0.21714724095162591;  // 1 / (2 ln 10)
#if defined(__HIP_DEVICE_COMPILE__)
    const double m = __builtin_amdgcn_frexp_mant(F);
    const int e = __builtin_amdgcn_frexp_exp(F);
#else
    int e = 0;
    const double m = std::frexp(F, &e);
    if (!(std::fabs(F) < HUGE_VAL)) e = 0;
#endif
    uint64_t u;
    std::memcpy(&u, &m, sizeof u);
    const LogBin b = tab[((uint32_t)(u >> 32) >> 12) & (kLogBins - 1)];
    const double r = fma(m, b.c, -1.0);
    const double p = fma(r, fma(r, fma(r, fma(r, H / 5, -H / 4), H / 3), -H / 2), H);
    return LogNorm{fma(r, p, b.l), e};
}

// log10 of the ratio of two norms. The exponents' difference is exact, so the result
// is as accurate for norms of any scale.
HM_LOGNORM_FN double log_ratio(const LogNorm &a, const LogNorm &b)
{
    return fma((double)(a.e - b.e), kHalfLog10Of2, a.f - b.f);
}

// The logarithm as one value, for the host check.
HM_LOGNORM_FN double half_log10(double F, const LogBin *tab)
{
    const LogNorm n = log_norm(F, tab);
    return fma((double)n.e, kHalfLog10Of2, n.f);
}

}  // namespace hm
