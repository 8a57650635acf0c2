// atan2 for the Birkhoff sums, by a table of atan(i / 64) in LDS: with ax = |x|,
// ay = |y|, mx and mn the larger and the smaller, i the nearest integer to
// 64 mn / mx and c = i / 64,
//   atan(mn / mx) = atan(c) + atan(u),  u = (mn - c mx) / (mx + c mn),  |u| <= 1/127,
// atan(u) by four terms of its series (the fifth is below 2e-18 u), then the octant
// and the signs, those of zeros included. Sums of magnitudes outside
// [2^-500, 2^500] (zero, subnormal, huge, infinite) are brought into range first, on
// a branch of the whole wavefront; NaN passes through (the lost lanes of a wavefront
// hold it, turn after turn). At most 7 units of 2^-53 of the result by its roundings,
// 3.2 found (tests/angle_check.cpp). About 45 instructions and three constants, where
// the library's takes about 65 and twenty, which the compiler keeps in registers
// through a loop.
// Compiles as host code too (no HIP types), so a host check can build it alone.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#define HM_ANGLE_FN __host__ __device__ inline
#else
#define HM_ANGLE_FN inline
#endif

namespace hm {

constexpr int kAngleBins = 65;

// atan(i / 64)
#if defined(__HIPCC__)
__device__
#endif
static const double kAtan[kAngleBins] = {
    0x0.0p+0, 0x1.fff555bbb729bp-7, 0x1.ffd55bba97625p-6, 0x1.7fb818430da2ap-5,
    0x1.ff55bb72cfdeap-5, 0x1.3f59f0e7c559dp-4, 0x1.7ee182602f10fp-4, 0x1.be39ebe6f07c3p-4,
    0x1.fd5ba9aac2f6ep-4, 0x1.1e1fafb043727p-3, 0x1.3d6eee8c6626cp-3, 0x1.5c9811e3ec26ap-3,
    0x1.7b97b4bce5b02p-3, 0x1.9a6a8e96c8626p-3, 0x1.b90d7529260a2p-3, 0x1.d77d5df205736p-3,
    0x1.f5b75f92c80ddp-3, 0x1.09dc597d86362p-2, 0x1.18bf5a30bf178p-2, 0x1.278372057ef46p-2,
    0x1.362773707ebccp-2, 0x1.44aa436c2af0ap-2, 0x1.530ad9951cd4ap-2, 0x1.614840309cfe2p-2,
    0x1.6f61941e4def1p-2, 0x1.7d5604b63b3f7p-2, 0x1.8b24d394a1b25p-2, 0x1.98cd5454d6b18p-2,
    0x1.a64eec3cc23fdp-2, 0x1.b3a911da65c6cp-2, 0x1.c0db4c94ec9f0p-2, 0x1.cde53432c1351p-2,
    0x1.dac670561bb4fp-2, 0x1.e77eb7f175a34p-2, 0x1.f40dd0b541418p-2, 0x1.0039c73c1a40cp-1,
    0x1.0657e94db30d0p-1, 0x1.0c6145b5b43dap-1, 0x1.1255d9bfbd2a9p-1, 0x1.1835a88be7c13p-1,
    0x1.1e00babdefeb4p-1, 0x1.23b71e2cc9e6ap-1, 0x1.2958e59308e31p-1, 0x1.2ee628406cbcap-1,
    0x1.345f01cce37bbp-1, 0x1.39c391cd4171ap-1, 0x1.3f13fb89e96f4p-1, 0x1.445065b795b56p-1,
    0x1.4978fa3269ee1p-1, 0x1.4e8de5bb6ec04p-1, 0x1.538f57b89061fp-1, 0x1.587d81f732fbbp-1,
    0x1.5d58987169b18p-1, 0x1.6220d115d7b8ep-1, 0x1.66d663923e087p-1, 0x1.6b798920b3d99p-1,
    0x1.700a7c5784634p-1, 0x1.748978fba8e0fp-1, 0x1.78f6bbd5d315ep-1, 0x1.7d528289fa093p-1,
    0x1.819d0b7158a4dp-1, 0x1.85d69576cc2c5p-1, 0x1.89ff5ff57f1f8p-1, 0x1.8e17aa99cc05ep-1,
    0x1.921fb54442d18p-1,
};

// Brings ax, ay into range with the same angle.
HM_ANGLE_FN void angle_rescale(double &ax, double &ay)
{
    const double s = ax + ay;
    if (s > 0x1p500) {
        const bool inf = !(ax < HUGE_VAL && ay < HUGE_VAL);
        ax = inf ? (ax < HUGE_VAL ? 0.0 : 1.0) : ax * 0x1p-600;
        ay = inf ? (ay < HUGE_VAL ? 0.0 : 1.0) : ay * 0x1p-600;
    } else if (s < 0x1p-500) {
        ax = s == 0.0 ? 1.0 : ax * 0x1p600;
        ay = ay * 0x1p600;
    }
}

// atan2(y, x); tab[i] = atan(i / 64).
HM_ANGLE_FN double angle_of(double y, double x, const double *tab)
{
    double ax = fabs(x), ay = fabs(y);
    const double s = ax + ay;
    const bool odd = s < 0x1p-500 || s > 0x1p500;
#if defined(__HIP_DEVICE_COMPILE__)
    if (__builtin_expect(__any(odd), 0)) angle_rescale(ax, ay);
#else
    if (odd) angle_rescale(ax, ay);
#endif
    const bool swap = ay > ax;
    const double mx = swap ? ay : ax, mn = swap ? ax : ay;
#if defined(__HIP_DEVICE_COMPILE__)
    const double q = mn * __builtin_amdgcn_rcp(mx);
#else
    const double q = mn / mx;
#endif
    const uint32_t i = q >= 0.0 ? (uint32_t)fma(q, 64.0, 0.5) : 0u;
    const double c = (double)i * (1.0 / 64.0);
    const double num = fma(-c, mx, mn), den = fma(c, mn, mx);
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(den);
#else
    double r = (double)(1.0f / (float)den);
    if (!(r > 0.0 && r < HUGE_VAL)) r = 1.0 / den;
#endif
    r = fma(fma(-den, r, 1.0), r, r);
    double u = num * r;
    u = fma(fma(-u, den, num), r, u);
    const double z = u * u;
    const double p = fma(z, fma(z, -1.0 / 7, 1.0 / 5), -1.0 / 3);
    const double a = tab[i > 64u ? 64u : i] + fma(u * z, p, u);
    // the octant: a, pi/2 - a, pi/2 + a or pi - a
    uint64_t xb;
    memcpy(&xb, &x, sizeof xb);
    const bool neg = xb >> 63;
    const double base = swap ? 1.57079632679489661923 : neg ? 3.14159265358979323846 : 0.0;
    return copysign(base + (swap != neg ? -a : a), y);
}

#if defined(__HIPCC__)
// Fills a workgroup's table of angle_of in LDS; every thread takes part, before a
// barrier of the caller's.
__device__ __forceinline__ void fill_angle_table(double *tab)
{
    for (int q = threadIdx.x; q < kAngleBins; q += blockDim.x) tab[q] = kAtan[q];
}
#endif

}  // namespace hm
