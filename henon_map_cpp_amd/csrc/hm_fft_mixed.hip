// FFT tunes of windows of any length (src/dynamic_indicator.cpp:32-61, 178-196,
// 255-331 for any N). Windows of up to about 10^4 points run in one kernel per
// signal with the whole signal in LDS (k_wh_tune, below the four-step
// kernels). Longer windows whose length has only the prime factors 2, 3, 5 and
// 7 run a mixed-radix four-step transform of the length itself, N = N1 x N2 (index n = N2 n1 + n2
// in, k = k1 + N1 k2 out):
//   X[k1 + N1 k2] = sum_{n2} W_{N2}^{n2 k2} W_N^{n2 k1} sum_{n1} x[N2 n1 + n2] W_{N1}^{n1 k1}
// with both factors LDS-resident, so no padding to a power of two and no chirp:
//   k_mr_columns : load, mean removal and Hanning of a few columns n2, N1-point
//                  FFTs, step twiddle W_N^{n2 k1}, store rows k1
//   k_mr_rows    : per row k1 the N2-point FFT, magnitudes (the spectrum's
//                  entry k1 + N1 k2 sits at k1 N2 + k2)
//   k_mr_tune    : per signal the first maximum in the spectrum's order and the
//                  three-point interpolation (dynamic_indicator.cpp:139-176)
// Sub-transforms are Stockham passes of radix 8, 4, 2, 3, 5, 7 (runtime plan)
// over several columns or rows per workgroup. HBM traffic per signal: the
// samples once, 16 N bytes of scratch each way, 8 N bytes of magnitudes each way.
//
// Other lengths run Bluestein's chirp-z transform over the smallest
// {2,3,5,7}-smooth length M >= 2N - 1 that splits the same way (with
// c_m = exp(-i pi m^2 / N): X_k = c_k sum_m (x_m c_m) conj(c_{k-m}), a cyclic
// convolution of length M with the fixed filter B = DFT_M(conj(c)), computed
// once per N on the host in long double). The same kernels with the chirp:
//   k_mr_columns<1> : chirped samples (zero from N on), M1-point FFTs, twiddle
//   k_mr_rows<1>    : per row k1 the M2-point FFT (the spectrum, entry
//                     k1 + M1 k2), times B, conjugate, M2-point FFT, twiddle
//                     W_M^{k1 j1}: the inverse transform as the conjugate of a
//                     forward one (input index k1 + M1 k2, output j1 + M2 j2)
//   k_mr_final      : per column j1 the M1-point FFT over k1 (giving j2), the
//                     magnitudes of the entries j = j1 + M2 j2 < N
//   k_mr_tune<1>    : first maximum and interpolation in natural order
// |X_k| = |conv_k| / M; the scale is left out since the first maximum and the
// interpolation (homogeneous of degree 0 in the magnitudes) do not see it.
// Windows too long for two 2048-point factors take the power-of-two chirp-z
// transform (hm_chirpz.hip).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdint>
#include <cstdlib>
#include <iterator>
#include <map>
#include <mutex>
#include <vector>

#include "hm_device.h"
#include "hm_internal.h"
#include "hm_tune.h"

namespace hm {

constexpr uint32_t kMrThreads = 512;
constexpr uint32_t kMrPmax = 2048;  // points of one workgroup's transforms (32 KiB)
constexpr int kMrMaxPasses = 12;

// Radix sequence of one sub-length, four bits per pass (pass s in bits 4s..4s+3):
// read by shifts, so no per-pass table is indexed at run time.
struct MrPlan {
    uint32_t L, n_pass;
    uint64_t radices;
};

struct MrArgs {
    const double *hist;
    HistLayout lay;
    const double *means;  // [4][n] or NULL
    uint32_t n, p0, nsig, from, N;
    uint32_t M;              // transform length: N, or the chirp-z length
    uint32_t N1, N2, C, RR;  // M = N1 x N2; C columns per workgroup (columns kernels), RR rows (rows kernel)
    MrPlan p1, p2;
    const double *hann;      // [N]
    const Cplx *tw1, *tw2;   // W_{N1}^q, W_{N2}^q
    const Cplx *twm;         // [N1][N2]: W_M^{k1 n2}
    const Cplx *chirp;       // chirp-z: [N] exp(-i pi (m^2 mod 2N) / N)
    const Cplx *bhat;        // chirp-z: [N1][N2], B[k1 + N1 k2] at k1 N2 + k2
    Cplx *Y;                 // scratch [nsig][N1][N2]
    double *mags;            // scratch [nsig][N]
    uint32_t *flags;         // [nsig]
    double *out;             // [window][plane][n]
    uint32_t window;
};

__device__ __forceinline__ void dft3(Cplx *v)
{
    // X1 = a + c (b + d) - i s (b - d), X2 = a + c (b + d) + i s (b - d)
    constexpr double c = -0.5, s = 0.86602540378443864676;  // cos, sin of 2 pi / 3
    const Cplx a = v[0], t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
    v[0] = cadd(a, t1);
    const Cplx m1 = Cplx{fma(c, t1.re, a.re), fma(c, t1.im, a.im)};
    const Cplx m2 = Cplx{s * t2.im, -(s * t2.re)};
    v[1] = cadd(m1, m2);
    v[2] = csub(m1, m2);
}

// cos and sin of 2 pi q / R for q = 1 .. (R-1)/2
template <int R>
__device__ __forceinline__ constexpr double root_cos(int q)
{
    if constexpr (R == 5) {
        constexpr double c[3] = {1.0, 0.30901699437494742408, -0.80901699437494742410};
        return c[q];
    } else if constexpr (R == 7) {
        constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440434, -0.90096886790241912632};
        return c[q];
    } else if constexpr (R == 11) {
        constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642549, -0.14231483827328514046,
                                 -0.65486073394528506413, -0.95949297361449738990};
        return c[q];
    } else {
        constexpr double c[7] = {1.0, 0.88545602565320989587, 0.56806474673115580249, 0.12053668025532305325,
                                 -0.35460488704253562600, -0.74851074817110109868, -0.97094181742605202719};
        return c[q];
    }
}
template <int R>
__device__ __forceinline__ constexpr double root_sin(int q)
{
    if constexpr (R == 5) {
        constexpr double s[3] = {0.0, 0.95105651629515357211, 0.58778525229247312913};
        return s[q];
    } else if constexpr (R == 7) {
        constexpr double s[4] = {0.0, 0.78183148246802980873, 0.97492791218182360698, 0.43388373911755812029};
        return s[q];
    } else if constexpr (R == 11) {
        constexpr double s[6] = {0.0, 0.54064081745559758210, 0.90963199535451837142, 0.98982144188093273236,
                                 0.75574957435425828370, 0.28173255684142969765};
        return s[q];
    } else {
        constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399284,
                                 0.93501624268541482345, 0.66312265824079520232, 0.23931566428755776695};
        return s[q];
    }
}

// Forward DFT of prime size R = 5, 7, 11, 13 from the pairs m, R - m: with
// a_m = v_m + v_{R-m}, b_m = v_m - v_{R-m} and t = 2 pi m k / R,
//   X_k = v_0 + sum_m (a_m cos t - i b_m sin t),  X_{R-k} = v_0 + sum_m (a_m cos t + i b_m sin t)
// (m, k = 1 .. (R-1)/2): (R-1) constants instead of (R-1)^2 products of roots.
template <int R>
__device__ __forceinline__ void dft_prime(Cplx *v)
{
    constexpr int H = (R - 1) / 2;
    Cplx a[H], b[H];
#pragma unroll
    for (int m = 1; m <= H; ++m) {
        a[m - 1] = cadd(v[m], v[R - m]);
        b[m - 1] = csub(v[m], v[R - m]);
    }
    Cplx x0 = v[0];
#pragma unroll
    for (int m = 0; m < H; ++m) x0 = cadd(x0, a[m]);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        Cplx p = v[0], q{0.0, 0.0};
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            const int r = (m * k) % R;
            const int f = r <= H ? r : R - r;  // cos t = cos(2 pi f / R), sin t = +-sin(2 pi f / R)
            const double c = root_cos<R>(f), sn = r <= H ? root_sin<R>(f) : -root_sin<R>(f);
            p.re = fma(a[m - 1].re, c, p.re);
            p.im = fma(a[m - 1].im, c, p.im);
            q.re = fma(b[m - 1].re, sn, q.re);
            q.im = fma(b[m - 1].im, sn, q.im);
        }
        // X_k = p - i q, X_{R-k} = p + i q
        v[k] = Cplx{p.re + q.im, p.im - q.re};
        v[R - k] = Cplx{p.re - q.im, p.im + q.re};
    }
    v[0] = x0;
}

template <int R>
__device__ __forceinline__ void dft_any(Cplx *v);

// 9 = 3 x 3 and 16 = 4 x 4: the inner DFTs over n1 of n = A n1 + n2, the roots
// W_R^{n2 k1}, the outer DFTs over n2 (k = k1 + A k2).
__device__ __forceinline__ void dft9(Cplx *v)
{
    // W_9^1, W_9^2, W_9^4
    constexpr Cplx w1{0.76604444311897803519, -0.64278760968653932633}, w2{0.17364817766693034880, -0.98480775301220805940},
        w4{-0.93969262078590838410, -0.34202014332566873297};
    Cplx a[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1) a[n2][n1] = v[3 * n1 + n2];
        dft3(a[n2]);
    }
    a[1][1] = cmul(a[1][1], w1);
    a[1][2] = cmul(a[1][2], w2);
    a[2][1] = cmul(a[2][1], w2);
    a[2][2] = cmul(a[2][2], w4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        Cplx b[3] = {a[0][k1], a[1][k1], a[2][k1]};
        dft3(b);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
    }
}
__device__ __forceinline__ void dft16(Cplx *v)
{
    constexpr double c1 = 0.92387953251128675610, s1 = 0.38268343236508977172, h = 0.70710678118654752440;
    Cplx a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < 4; ++n1) a[n2][n1] = v[4 * n1 + n2];
        dft4(a[n2][0], a[n2][1], a[n2][2], a[n2][3]);
    }
    // W_16^q: q = 1, 2, 3 (n2 = 1), 2, 4, 6 (n2 = 2), 3, 6, 9 (n2 = 3)
    a[1][1] = cmul(a[1][1], Cplx{c1, -s1});
    a[1][2] = Cplx{h * (a[1][2].re + a[1][2].im), h * (a[1][2].im - a[1][2].re)};
    a[1][3] = cmul(a[1][3], Cplx{s1, -c1});
    a[2][1] = Cplx{h * (a[2][1].re + a[2][1].im), h * (a[2][1].im - a[2][1].re)};
    a[2][2] = mul_mi(a[2][2]);
    a[2][3] = Cplx{h * (a[2][3].im - a[2][3].re), -h * (a[2][3].re + a[2][3].im)};
    a[3][1] = cmul(a[3][1], Cplx{s1, -c1});
    a[3][2] = Cplx{h * (a[3][2].im - a[3][2].re), -h * (a[3][2].re + a[3][2].im)};
    a[3][3] = cmul(a[3][3], Cplx{-c1, s1});
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        dft4(a[0][k1], a[1][k1], a[2][k1], a[3][k1]);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = a[k2][k1];
    }
}

// R = A B with coprime factors: n = (B n1 + A n2) mod R, k the number with
// k mod A = k1 and k mod B = k2; no roots between the two steps.
template <int A, int B>
__device__ __forceinline__ void dft_coprime(Cplx *v)
{
    constexpr int R = A * B;
    Cplx t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % R];
        dft_any<A>(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        Cplx b[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) b[n2] = t[n2][k1];
        dft_any<B>(b);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) {
            int k = k1;
            while (k % B != k2) k += A;
            v[k] = b[k2];
        }
    }
}

template <int R>
__device__ __forceinline__ void dft_any(Cplx *v)
{
    if constexpr (R == 2 || R == 4 || R == 8) dft_r<R>(v);
    else if constexpr (R == 3) dft3(v);
    else if constexpr (R == 6) dft_coprime<2, 3>(v);
    else if constexpr (R == 9) dft9(v);
    else if constexpr (R == 10) dft_coprime<2, 5>(v);
    else if constexpr (R == 12) dft_coprime<4, 3>(v);
    else if constexpr (R == 16) dft16(v);
    else dft_prime<R>(v);
}

// LDS position of entry i of a signal: one pad entry after every 16, so that
// the power-of-two strides of the early passes' stores (R entries of 16 bytes
// apart when Ns = 1) fall into distinct banks.
__device__ __forceinline__ uint32_t lp(uint32_t i) { return i + (i >> 4); }
// LDS entries a signal of L entries spans (lp(L - 1) + 1); the odd variant for
// the columns kernels, whose loads step across signals.
__host__ __device__ constexpr uint32_t lds_len(uint32_t L) { return L + (L - 1) / 16 + 1; }
__host__ __device__ constexpr uint32_t lds_len_odd(uint32_t L) { return lds_len(L) | 1u; }

// One radix-R Stockham pass over G signals of length L in LDS (signal g at
// buf[g GS ..], entry i at lp(i)); Ns = product of the earlier radices. Butterfly j reads
// x[j + r L/R], twiddles by W_L^{k r L/(Ns R)} (k = j mod Ns; one table load, the
// higher powers by products), takes the R-point DFT and writes element r to
// (j - k) R + k + r Ns.
template <int R>
__device__ __forceinline__ void mr_pass(Cplx *buf, uint32_t G, uint32_t L, uint32_t GS, uint32_t Ns,
                                        const Cplx *__restrict__ tw)
{
    constexpr uint32_t PER = (kMrPmax / R + kMrThreads - 1) / kMrThreads;
    const uint32_t B = L / R, total = G * B, step = L / (Ns * R);
    Cplx v[PER][R];
    uint32_t goff[PER], base[PER];
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        const uint32_t J = threadIdx.x + q * kMrThreads;
        base[q] = 0xffffffffu;
        if (J < total) {
            const uint32_t g = J / B, j = J - g * B;
            const Cplx *src = buf + g * GS;
#pragma unroll
            for (int r = 0; r < R; ++r) v[q][r] = src[lp(j + r * B)];
            const uint32_t k = j % Ns;
            if (k != 0) {
                const Cplx w1 = tw[k * step];
                Cplx w = w1;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    v[q][r] = cmul(v[q][r], w);
                    if (r + 1 < R) w = cmul(w, w1);
                }
            }
            dft_any<R>(v[q]);
            goff[q] = g * GS;
            base[q] = (j - k) * R + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        if (base[q] != 0xffffffffu) {
            Cplx *dst = buf + goff[q];
            const uint32_t ns = Ns;
#pragma unroll
            for (int r = 0; r < R; ++r) dst[lp(base[q] + r * ns)] = v[q][r];
        }
    }
    __syncthreads();
}

// Forward DFT of G signals of length p.L in LDS, in natural order.
__device__ __forceinline__ void mr_fft(Cplx *buf, uint32_t G, const MrPlan &p, uint32_t GS, const Cplx *__restrict__ tw)
{
    uint32_t Ns = 1;
    for (uint32_t s = 0; s < p.n_pass; ++s) {
        const uint32_t R = (uint32_t)(p.radices >> (4 * s)) & 15u;
        switch (R) {
        case 8: mr_pass<8>(buf, G, p.L, GS, Ns, tw); break;
        case 4: mr_pass<4>(buf, G, p.L, GS, Ns, tw); break;
        case 2: mr_pass<2>(buf, G, p.L, GS, Ns, tw); break;
        case 3: mr_pass<3>(buf, G, p.L, GS, Ns, tw); break;
        case 5: mr_pass<5>(buf, G, p.L, GS, Ns, tw); break;
        default: mr_pass<7>(buf, G, p.L, GS, Ns, tw); break;
        }
        Ns *= R;
    }
}

__device__ __forceinline__ uint32_t mr_virtual(uint32_t b, uint32_t per) { return (b % 8) * per + b / 8; }

template <bool CZ>
__global__ void __launch_bounds__(kMrThreads, 4) k_mr_columns(MrArgs a)
{
    extern __shared__ Cplx buf[];
    const uint32_t per_sig = a.N2 / a.C;
    const uint32_t total = a.nsig * per_sig;
    const uint32_t v = mr_virtual(blockIdx.x, gridDim.x / 8);
    if (v >= total) return;
    const uint32_t sig = v / per_sig, c0 = (v % per_sig) * a.C;
    const uint32_t C = a.C, N1 = a.N1, N2 = a.N2, GS = lds_len_odd(N1);
    const uint32_t particle = a.p0 + sig / 2, plane = sig % 2;
    const size_t nn = a.n;
    double mc[4] = {0.0, 0.0, 0.0, 0.0};
    if (a.means)
        for (int c = 0; c < 4; ++c) mc[c] = a.means[c * nn + particle];
    if (any_nan(mc[0], mc[1], mc[2], mc[3])) {
        // a NaN mean makes every sample of its coordinate NaN: nothing to read
        if (threadIdx.x == 0) atomicOr(a.flags + sig, 1u);
        return;
    }
    // four finite means prove that no sample of the particle is NaN or
    // infinite: the other plane need not be read
    const bool scan_other =
        !a.means || !(isfinite(mc[0]) && isfinite(mc[1]) && isfinite(mc[2]) && isfinite(mc[3]));
    const int cx = 2 * plane, cp = cx + 1, co0 = 2 * (1 - plane), co1 = co0 + 1;
    bool nan_seen = false;
    for (uint32_t e = threadIdx.x; e < C * N1; e += kMrThreads) {
        const uint32_t n1 = e / C, c = e - n1 * C;
        const uint32_t m = n1 * N2 + c0 + c;
        Cplx z{0.0, 0.0};
        if (!CZ || m < a.N) {
            const uint64_t sm = (uint64_t)a.from + m;
            const double vx = a.hist[hat(a.lay, sm, cx, particle)] - mc[cx];
            const double vp = a.hist[hat(a.lay, sm, cp, particle)] - mc[cp];
            nan_seen |= __builtin_isnan(vx) || __builtin_isnan(vp);
            if (scan_other)
                nan_seen |= __builtin_isnan(a.hist[hat(a.lay, sm, co0, particle)] - mc[co0]) ||
                            __builtin_isnan(a.hist[hat(a.lay, sm, co1, particle)] - mc[co1]);
            const double h = a.hann[m];
            z = Cplx{vx * h, vp * h};
            if constexpr (CZ) z = cmul(z, a.chirp[m]);
        }
        buf[c * GS + lp(n1)] = z;
    }
    if (__any(nan_seen) && (threadIdx.x & 63) == 0) atomicOr(a.flags + sig, 1u);
    __syncthreads();
    mr_fft(buf, C, a.p1, GS, a.tw1);
    Cplx *Y = a.Y + (size_t)sig * a.M;
    for (uint32_t e = threadIdx.x; e < C * N1; e += kMrThreads) {
        const uint32_t k1 = e / C, c = e - k1 * C;
        const size_t o = (size_t)k1 * N2 + c0 + c;
        Y[o] = cmul(buf[c * GS + lp(k1)], a.twm[o]);
    }
}

template <bool CZ>
__global__ void __launch_bounds__(kMrThreads, 4) k_mr_rows(MrArgs a)
{
    extern __shared__ Cplx buf[];
    const uint32_t per_sig = a.N1 / a.RR;
    const uint32_t total = a.nsig * per_sig;
    const uint32_t v = mr_virtual(blockIdx.x, gridDim.x / 8);
    if (v >= total) return;
    const uint32_t sig = v / per_sig, r0 = (v % per_sig) * a.RR;
    const uint32_t N2 = a.N2, P = a.RR * N2, GS = lds_len(N2);
    // row g entry i (global offset e = g N2 + i) at LDS g GS + lp(i)
    auto at = [&](uint32_t e) {
        const uint32_t g = e / N2;
        return g * GS + lp(e - g * N2);
    };
    Cplx *Y = a.Y + (size_t)sig * a.M + (size_t)r0 * N2;
    for (uint32_t e = threadIdx.x; e < P; e += kMrThreads) buf[at(e)] = Y[e];
    __syncthreads();
    mr_fft(buf, a.RR, a.p2, GS, a.tw2);
    if constexpr (CZ) {
        // spectrum entry k1 + N1 k2 times B, conjugated: the inverse transform
        // becomes a forward one over k2 (then k1, in k_mr_final)
        const Cplx *bh = a.bhat + (size_t)r0 * N2;
        for (uint32_t e = threadIdx.x; e < P; e += kMrThreads) {
            const uint32_t l = at(e);
            const Cplx z = cmul(buf[l], bh[e]);
            buf[l] = Cplx{z.re, -z.im};
        }
        __syncthreads();
        mr_fft(buf, a.RR, a.p2, GS, a.tw2);
        const Cplx *tm = a.twm + (size_t)r0 * N2;
        for (uint32_t e = threadIdx.x; e < P; e += kMrThreads) Y[e] = cmul(buf[at(e)], tm[e]);
    } else {
        // spectrum entry k1 + N1 k2 at row k1, position k2
        double *mags = a.mags + (size_t)sig * a.N + (size_t)r0 * N2;
        for (uint32_t e = threadIdx.x; e < P; e += kMrThreads) {
            const Cplx z = buf[at(e)];
            mags[e] = sqrt(z.re * z.re + z.im * z.im);
        }
    }
}

// Chirp-z only: columns j1 in [c0, c0 + C), the M1-point transforms over k1
// (output j2) and the magnitudes of the entries j = j1 + N2 j2 < N.
__global__ void __launch_bounds__(kMrThreads, 4) k_mr_final(MrArgs a)
{
    extern __shared__ Cplx buf[];
    const uint32_t per_sig = a.N2 / a.C;
    const uint32_t total = a.nsig * per_sig;
    const uint32_t v = mr_virtual(blockIdx.x, gridDim.x / 8);
    if (v >= total) return;
    const uint32_t sig = v / per_sig, c0 = (v % per_sig) * a.C;
    const uint32_t C = a.C, N1 = a.N1, N2 = a.N2, GS = lds_len_odd(N1);
    const Cplx *Y = a.Y + (size_t)sig * a.M;
    for (uint32_t e = threadIdx.x; e < C * N1; e += kMrThreads) {
        const uint32_t k1 = e / C, c = e - k1 * C;
        buf[c * GS + lp(k1)] = Y[(size_t)k1 * N2 + c0 + c];
    }
    __syncthreads();
    mr_fft(buf, C, a.p1, GS, a.tw1);
    double *mags = a.mags + (size_t)sig * a.N;
    for (uint32_t e = threadIdx.x; e < C * N1; e += kMrThreads) {
        const uint32_t j2 = e / C, c = e - j2 * C;
        const uint32_t j = c0 + c + j2 * N2;
        if (j < a.N) {
            const Cplx z = buf[c * GS + lp(j2)];
            mags[j] = sqrt(z.re * z.re + z.im * z.im);
        }
    }
}

template <bool NATURAL>
__global__ void __launch_bounds__(kMrThreads) k_mr_tune(MrArgs a)
{
    __shared__ double sv[kMrThreads / 64];
    __shared__ uint32_t si[kMrThreads / 64];
    const uint32_t sig = blockIdx.x;
    if (sig >= a.nsig) return;
    const uint32_t particle = a.p0 + sig / 2, plane = sig % 2;
    double *o = a.out + ((size_t)a.window * 2 + plane) * a.n + particle;
    if (a.flags[sig]) {
        if (threadIdx.x == 0) *o = __builtin_nan("");
        return;
    }
    const double *mags = a.mags + (size_t)sig * a.N;
    const uint32_t N1 = a.N1, N2 = a.N2;
    // first maximum in the spectrum's order: the lowest k among equal
    // magnitudes, whatever the storage order (k1 N2 + k2 for k = k1 + N1 k2)
    double v = -1.0;
    uint32_t i = 0xffffffffu;
    for (uint32_t p = threadIdx.x; p < a.N; p += kMrThreads) {
        const double mg = mags[p];
        uint32_t k = p;
        if constexpr (!NATURAL) {
            const uint32_t k1 = p / N2;
            k = k1 + N1 * (p - k1 * N2);
        }
        if (mg > v || (mg == v && k < i) || i == 0xffffffffu) { v = mg; i = k; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double ov = __shfl_xor(v, off);
        const uint32_t oi = __shfl_xor(i, off);
        if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
    }
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = v; si[threadIdx.x >> 6] = i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double bv = sv[0];
        uint32_t bi = si[0];
        for (uint32_t q = 1; q < kMrThreads / 64; ++q)
            if (sv[q] > bv || (sv[q] == bv && si[q] < bi)) { bv = sv[q]; bi = si[q]; }
        if constexpr (NATURAL) *o = interp_tune_at([&](uint32_t k) { return mags[k]; }, a.N, bi);
        else *o = interp_tune_at([&](uint32_t k) { return mags[(size_t)(k % N1) * N2 + k / N1]; }, a.N, bi);
    }
}

// ---------------------------------------------------------------- whole-signal transforms
// A window whose transform length fits one workgroup's LDS (about 10^4 points
// in 160 KiB) runs in one kernel, one workgroup per signal: the samples are
// read once, every pass runs in LDS and the tune is found there, with no
// scratch in HBM and no second launch.
//   direct : lengths whose prime factors are 2 to 13 (passes of radix 2 to 13 and
//            16 in registers) or other primes up to kWhPrimeMax (one pass each,
//            on the matrix cores where it fits them)
//   chirp-z: other lengths N, over a smooth M >= 2N - 1 that fits: the chirped
//            samples, FFT_M, times B = DFT_M(conj(c)), conjugated, FFT_M again;
//            |X_k| = |V_k| / M for k < N (the scale does not change the tune)
// The signal sits in LDS unpadded: the first pass takes an odd radix where the
// length has an odd factor, so its stores step by an odd number of 16-byte
// entries, and the later passes store runs of consecutive entries (a power of
// two pays some bank conflicts in its first pass).
// At 10^4 points one workgroup has the CU to itself and runs the phases one after
// the other, in cycles: the load 15000 (12000 with the chip idle: the CU's own way
// to L2), a radix-10 pass 6000 (320 KB through LDS 2500, 60 FP64 instructions per
// point and wavefront 3700), the maximum and the tune 7000. 10000 points as 10^4
// instead of 5^4 x 2 x 8, twiddles read in order instead of strided through one
// table (64 cache lines an instruction) and one square root a signal instead of
// one an entry: 129 -> 91 ns per signal; 500 points (10 x 10 x 5, one wavefront)
// 7.7 -> 3.1, 501 (chirp-z over 7 x 9 x 16 instead of 3 x 3 x 7 x 2 x 8) 16.3 -> 11.
// Samples by stepped pointers instead of an address formed of three products each:
// 91 -> 84 ns, 500 points 3.1 -> 2.8.
// The shapes of k_wh_tune: 64, 128 .. kWhThreads threads for up to ten points a
// thread (a butterfly of the radix-10 passes each, every wavefront at work; 16
// wavefronts and up to 160 KiB of signals per CU in every shape).
constexpr uint32_t kWhThreads = 1024, kWhPoints = 10, kWhPmax = kWhPoints * kWhThreads;
constexpr uint32_t kWhPrimeMax = 257;
constexpr int kWhMaxPasses = 16;

// One pass: radix R after the radices of product Ns, B = L / R butterflies; tw =
// where its twiddles start in the plan's table, in the order that the butterflies
// read them (k = 0 .. Ns - 1 of W_{Ns R}^k, or for a prime pass the rows r = 1 ..
// R - 1 of W_{Ns R}^{r k}; none if Ns = 1); m_* are the multipliers of udiv_m for
// Ns, B and (R + 1) / 2; frag = where the root matrix of a matrix pass starts in
// the plan's (kNoFrag: another pass), root = where W_R^q of another prime pass
// starts in the table.
constexpr uint32_t kNoFrag = 0xffffffffu;
struct WhPass {
    uint32_t R, Ns, B, tw, m_ns, m_b, m_h1, frag, root;
};
struct WhPlan {
    uint32_t L, n_pass;
    WhPass pass[kWhMaxPasses];
};

// j / d for j < 2^16 and d <= 2^16 from m = floor(2^32 / d) + 1 (m = 0: d = 1):
// j m / 2^32 = j / d + j (m - 2^32 / d) / 2^32 exceeds j / d by less than
// 2^-16, and the fraction of j / d is at most 1 - 1 / d.
__device__ __forceinline__ uint32_t udiv_m(uint32_t j, uint32_t m) { return m ? __umulhi(j, m) : j; }

struct WhArgs {
    const double *hist;
    HistLayout lay;
    const double *means;  // [4][n] or NULL
    uint32_t n, p0, from, N, M;
    WhPlan plan;          // passes of the M-point transform
    const double *hann;   // [N]
    const Cplx *tw;       // the passes' twiddles
    const Cplx *frag;     // the root matrices of the matrix passes
    const Cplx *chirp;    // chirp-z: [N]
    const Cplx *bhat;     // chirp-z: [M], B in natural order
    double *out;          // [window][plane][n]
    uint32_t window;
    double cos_n, sin_n;  // of 2 pi / N
};

// One radix-R Stockham pass (as mr_pass) over the whole signal of length L:
// butterfly j reads x[j + r L/R], twiddles by W_{Ns R}^{k r} (k = j mod Ns; one
// load, neighbours from neighbours, the powers by products), takes the R-point
// DFT and writes element r to (j - k) R + k + r Ns.
template <int R, uint32_t NT, uint32_t PMAX>
__device__ __forceinline__ void wh_pass(Cplx *buf, const WhPass &ps, const Cplx *__restrict__ tws)
{
    constexpr uint32_t PER = (PMAX / R + NT - 1) / NT;
    const uint32_t B = ps.B, Ns = ps.Ns;
    const Cplx *tw = tws + ps.tw;
    Cplx v[PER][R];
    uint32_t base[PER];
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        const uint32_t j = threadIdx.x + q * NT;
        base[q] = 0xffffffffu;
        if (j < B) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[q][r] = buf[j + r * B];
            const uint32_t k = j - udiv_m(j, ps.m_ns) * Ns;
            if (Ns > 1) {
                Cplx w[R];
                w[1] = tw[k];
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    if (r > 1) w[r] = r % 2 ? cmul(w[r - 1], w[1]) : cmul(w[r / 2], w[r / 2]);
                    v[q][r] = cmul(v[q][r], w[r]);
                }
            }
            dft_any<R>(v[q]);
            base[q] = (j - k) * R + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q)
        if (base[q] != 0xffffffffu)
#pragma unroll
            for (int r = 0; r < R; ++r) buf[base[q] + r * Ns] = v[q][r];
    __syncthreads();
}

// A pass of odd prime radix R (17 .. kWhPrimeMax) takes the R-point DFT from the
// pairs (r, R - r) as in dft_prime, H = (R - 1) / 2:
//   fold : each pair twiddled and replaced in place by a_r = x_r + x_{R-r} (at r)
//          and b_r = x_r - x_{R-r} (at R - r)
//   sums : Y_q = x_0 + sum_r (a_r cos t - i b_r sin t), Y_{R-q} with + i, t = 2 pi r q / R,
//          for q = 0 .. H (q = 0: the sum alone)
template <uint32_t NT>
__device__ __forceinline__ void wh_fold_pairs(Cplx *buf, const WhPass &ps, const Cplx *__restrict__ tws)
{
    const uint32_t R = ps.R, Ns = ps.Ns, B = ps.B, H = (R - 1) / 2;
    const Cplx *tw = tws + ps.tw;
    for (uint32_t e = threadIdx.x; e < B * H; e += NT) {
        const uint32_t r0 = udiv_m(e, ps.m_b), r = r0 + 1, j = e - r0 * B, k = j - udiv_m(j, ps.m_ns) * Ns;
        const uint32_t iu = j + r * B, iv = j + (R - r) * B;
        Cplx u = buf[iu], v = buf[iv];
        if (Ns > 1) {
            u = cmul(u, tw[r0 * Ns + k]);
            v = cmul(v, tw[(R - 1 - r) * Ns + k]);
        }
        buf[iu] = cadd(u, v);
        buf[iv] = csub(u, v);
    }
    __syncthreads();
}

// The sums as matrix products on the matrix cores: the roots' cosines and sines
// (rows q, columns r) times the a_r and b_r of 16 butterflies, real and
// imaginary parts apart, v_mfma_f64_16x16x4 each. A wavefront takes up to
// kMatrixRounds tiles of 16 outputs by 16 butterflies and keeps their sums in
// registers until every wavefront has read its terms. The vector form reads both
// terms for every output (bound by LDS) and computes its roots; here a term serves
// 16 outputs and the matrix cores set the pace: of 101000 cycles at 10001 = 73 x 137
// points the two products take 20000 and 36000, where the instructions alone would
// (padding to 16 included) 16000 and 30000. 10001 points 331 -> 184 ns per signal
// (171 with the load's pointers stepped).
constexpr uint32_t kMatrixRounds = 2;
using Quad = double __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr uint32_t matrix_steps(uint32_t R) { return ((R - 1) / 2 + 3) / 4; }
__host__ __device__ constexpr uint32_t matrix_rows(uint32_t R) { return ((R - 1) / 2 + 16) / 16; }
__host__ __device__ constexpr uint32_t matrix_tiles(uint32_t R, uint32_t B) { return matrix_rows(R) * ((B + 15) / 16); }

template <uint32_t NT>
__device__ __forceinline__ void wh_pass_matrix(Cplx *buf, const WhPass &ps, const Cplx *__restrict__ tw,
                                               const Cplx *__restrict__ frags)
{
    wh_fold_pairs<NT>(buf, ps, tw);
    const uint32_t R = ps.R, Ns = ps.Ns, B = ps.B, H = (R - 1) / 2;
    const uint32_t steps = matrix_steps(R), rows = matrix_rows(R), tiles = matrix_tiles(R, B);
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = lane & 15, sub = lane >> 4;
    Quad cr[kMatrixRounds], ci[kMatrixRounds], sr[kMatrixRounds], si[kMatrixRounds];
#pragma unroll
    for (uint32_t g = 0; g < kMatrixRounds; ++g) {
        sr[g] = si[g] = Quad{0.0, 0.0, 0.0, 0.0};
        const uint32_t tile = wave + g * (NT / 64);
        if (tile >= tiles) continue;
        const uint32_t ct = tile / rows, rt = tile - ct * rows;
        const uint32_t j = min(ct * 16 + col, B - 1);
        const Cplx x0 = buf[j];
        cr[g] = Quad{x0.re, x0.re, x0.re, x0.re};
        ci[g] = Quad{x0.im, x0.im, x0.im, x0.im};
        const Cplx *f = frags + ps.frag + (size_t)rt * steps * 64 + lane;
        // terms r = 4 t + sub + 1, a_r and b_r of the lane's butterfly (zero beyond
        // H, which only the last step reaches), requested a step ahead of their use
        struct Term {
            Cplx w, a, b;
        };
        const Cplx *pa = buf + j + (sub + 1) * B, *pb = buf + j + (R - 1 - sub) * B;
        auto term = [&](uint32_t t) {
            Term m{f[t * 64], pa[t * 4 * B], pb[-(int)(t * 4 * B)]};
            if (t + 1 == steps && t * 4 + sub + 1 > H) m.a = m.b = Cplx{0.0, 0.0};
            return m;
        };
        auto add = [&](const Term &m) {
            cr[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(m.w.re, m.a.re, cr[g], 0, 0, 0);
            ci[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(m.w.re, m.a.im, ci[g], 0, 0, 0);
            sr[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(m.w.im, m.b.re, sr[g], 0, 0, 0);
            si[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(m.w.im, m.b.im, si[g], 0, 0, 0);
        };
        Term even = term(0);
        uint32_t t = 0;
        for (; t + 2 <= steps; t += 2) {
            const Term odd = term(t + 1);
            add(even);
            even = term(min(t + 2, steps - 1));
            add(odd);
        }
        if (t < steps) add(even);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t g = 0; g < kMatrixRounds; ++g) {
        const uint32_t tile = wave + g * (NT / 64);
        if (tile >= tiles) continue;
        const uint32_t ct = tile / rows, rt = tile - ct * rows, j = ct * 16 + col;
        const uint32_t k = j - udiv_m(j, ps.m_ns) * Ns, ob = (j - k) * R + k;
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            // the lane's sums: rows 4 e + sub of the tile
            const uint32_t q = rt * 16 + 4 * e + sub;
            if (j < B && q <= H) {
                buf[ob + q * Ns] = Cplx{cr[g][e] + si[g][e], ci[g][e] - sr[g][e]};
                if (q > 0) buf[ob + (R - q) * Ns] = Cplx{cr[g][e] - si[g][e], ci[g][e] + sr[g][e]};
            }
        }
    }
    __syncthreads();
}

// The sums of a pass without a root matrix: one thread per output pair
// (q, R - q) of a butterfly; the lanes of a wavefront share the butterfly (the
// same a_r, b_r: LDS broadcasts) and step cos t, sin t by the three-term
// recurrence f(r+1) = 2 cos(2 pi q / R) f(r) - f(r-1) (two multiply-adds a
// step). The recurrence's rounding errors grow at most like
// r min(r, 1 / |sin(2 pi q / R)|) units in the last place: about 1e-12 of the
// unit roots at most over the (R-1)/2 <= 128 steps, far under what moves a
// tune (the tests hold the tunes to 1e-12 of the long-double DFT's).
template <uint32_t NT, uint32_t PMAX>
__device__ __forceinline__ void wh_pass_prime(Cplx *buf, const WhPass &ps, const Cplx *__restrict__ tw)
{
    // output pairs per thread: B (H + 1) <= L (R + 1) / (2R) <= 0.55 L for R >= 11
    constexpr uint32_t GP = ((PMAX * 11 / 20 + NT - 1) / NT + 1) / 2 * 2;
    const uint32_t R = ps.R, Ns = ps.Ns, B = ps.B, H = (R - 1) / 2;
    wh_fold_pairs<NT>(buf, ps, tw);
    // output positions (< 2^15) of Y_q in the low, of Y_{R-q} in the high half
    static_assert(PMAX < 0xffffu, "output positions are packed in 16 bits");
    static_assert(GP % 2 == 0, "output pairs are taken two at a time");
    Cplx y0[GP], y1[GP];
    uint32_t oo[GP];
    const uint32_t items = B * (H + 1);
#pragma unroll
    for (uint32_t g = 0; g < GP; g += 2) {
        // two output pairs at once (independent chains); q = 0 runs the same
        // loop with cos = 1, sin = 0, which leaves Y_0 = x_0 + sum a_r
        uint32_t ja[2], qa[2];
        Cplx pa[2], sb[2];
        double c[2], sn[2], cp[2], sp[2], t2[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t e = min(threadIdx.x + (g + h) * NT, items - 1);
            ja[h] = udiv_m(e, ps.m_h1);
            qa[h] = e - ja[h] * (H + 1);
            const Cplx wq = tw[ps.root + qa[h]];  // exp(-2 pi i q / R)
            c[h] = wq.re;
            sn[h] = -wq.im;
            cp[h] = 1.0;
            sp[h] = 0.0;
            t2[h] = 2.0 * wq.re;
            pa[h] = buf[ja[h]];
            sb[h] = Cplx{0.0, 0.0};
        }
        for (uint32_t r = 1; r <= H; ++r) {
            Cplx av[2], bv[2];
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                av[h] = buf[ja[h] + r * B];
                bv[h] = buf[ja[h] + (R - r) * B];
            }
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                pa[h].re = fma(av[h].re, c[h], pa[h].re);
                pa[h].im = fma(av[h].im, c[h], pa[h].im);
                sb[h].re = fma(bv[h].re, sn[h], sb[h].re);
                sb[h].im = fma(bv[h].im, sn[h], sb[h].im);
                // cos, sin of (r + 1) 2 pi q / R: f(r+1) = 2 cos(2 pi q / R) f(r) - f(r-1)
                const double cn = fma(t2[h], c[h], -cp[h]), sn2 = fma(t2[h], sn[h], -sp[h]);
                cp[h] = c[h];
                sp[h] = sn[h];
                c[h] = cn;
                sn[h] = sn2;
            }
        }
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t e = threadIdx.x + (g + h) * NT;
            const uint32_t k = ja[h] - udiv_m(ja[h], ps.m_ns) * Ns, ob = (ja[h] - k) * R + k, q = qa[h];
            y0[g + h] = Cplx{pa[h].re + sb[h].im, pa[h].im - sb[h].re};  // Y_q
            y1[g + h] = Cplx{pa[h].re - sb[h].im, pa[h].im + sb[h].re};  // Y_{R-q}
            oo[g + h] = e >= items ? 0xffffffffu
                        : q == 0   ? (0xffff0000u | ob)
                                   : ((ob + q * Ns) | ((ob + (R - q) * Ns) << 16));
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t g = 0; g < GP; ++g) {
        const uint32_t lo = oo[g] & 0xffffu, hi = oo[g] >> 16;
        if (lo != 0xffffu) buf[lo] = y0[g];
        if (hi != 0xffffu) buf[hi] = y1[g];
    }
    __syncthreads();
}

// Forward DFT of the whole signal in LDS, in natural order. The plan lists its
// radices grouped as here (an odd or small first radix keeps the first pass's
// strided stores off shared banks), so each radix gets a loop of its own: one
// switch over the inlined passes inside a single loop keeps more registers live
// than any pass needs.
template <uint32_t NT, uint32_t PMAX>
__device__ __forceinline__ void wh_fft(Cplx *buf, const WhPlan &p, const Cplx *__restrict__ tw,
                                       const Cplx *__restrict__ frags)
{
    uint32_t s = 0;
    for (; s < p.n_pass && p.pass[s].R == 3; ++s) wh_pass<3, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 5; ++s) wh_pass<5, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 7; ++s) wh_pass<7, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 9; ++s) wh_pass<9, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 11; ++s) wh_pass<11, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 13; ++s) wh_pass<13, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R > 16; ++s) {
        if (p.pass[s].frag != kNoFrag) wh_pass_matrix<NT>(buf, p.pass[s], tw, frags);
        else wh_pass_prime<NT, PMAX>(buf, p.pass[s], tw);
    }
    for (; s < p.n_pass && p.pass[s].R == 6; ++s) wh_pass<6, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 10; ++s) wh_pass<10, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 2; ++s) wh_pass<2, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 12; ++s) wh_pass<12, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 4; ++s) wh_pass<4, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 8; ++s) wh_pass<8, NT, PMAX>(buf, p.pass[s], tw);
    for (; s < p.n_pass && p.pass[s].R == 16; ++s) wh_pass<16, NT, PMAX>(buf, p.pass[s], tw);
}

// One workgroup per signal (2 per particle: plane x, plane y): load, mean
// removal and Hanning, the transform(s), the first maximum of |X_k| over
// k < N and the three-point interpolation (dynamic_indicator.cpp:139-196).
template <bool CZ, uint32_t NT>
__global__ void __launch_bounds__(NT, 4) k_wh_tune(WhArgs a)
{
    constexpr uint32_t PMAX = kWhPoints * NT;
    extern __shared__ Cplx buf[];
    __shared__ double sv[NT / 64];
    __shared__ uint32_t first;
    const uint32_t sig = blockIdx.x;
    const uint32_t particle = a.p0 + sig / 2, plane = sig % 2;
    const size_t nn = a.n;
    double *o = a.out + ((size_t)a.window * 2 + plane) * nn + particle;
    const uint32_t N = a.N, M = a.M;
    double mc[4] = {0.0, 0.0, 0.0, 0.0};
    if (a.means)
        for (int c = 0; c < 4; ++c) mc[c] = a.means[c * nn + particle];
    if (any_nan(mc[0], mc[1], mc[2], mc[3])) {
        // a NaN mean makes every sample of its coordinate NaN: nothing to read
        if (threadIdx.x == 0) *o = __builtin_nan("");
        return;
    }
    // four finite means prove that no sample of the particle is NaN or
    // infinite: the other plane need not be read
    const bool scan_other =
        !a.means || !(isfinite(mc[0]) && isfinite(mc[1]) && isfinite(mc[2]) && isfinite(mc[3]));
    const int cx = 2 * plane, cp = cx + 1, co0 = 2 * (1 - plane), co1 = co0 + 1;
    // selected once: an index into mc at run time is a chain of compares at each use
    const double mean_x = plane ? mc[2] : mc[0], mean_p = plane ? mc[3] : mc[1];
    const double mean_o0 = plane ? mc[0] : mc[2], mean_o1 = plane ? mc[1] : mc[3];
    int nan_seen = 0;
    // every sample load of the thread issued before the first use (a loop
    // that waits for each sample in turn leaves the workgroup idle)
    constexpr uint32_t LP = (CZ ? PMAX / 2 : PMAX + NT - 1) / NT + (CZ ? 1 : 0);
    double vx[LP], vp[LP], hh[LP];
    const double *px = a.hist + hat(a.lay, (uint64_t)a.from + threadIdx.x, cx, particle);
    const size_t to_p = a.lay.cs, ahead = (size_t)NT * a.lay.ms;
#pragma unroll
    for (uint32_t u = 0; u < LP; ++u) {
        const uint32_t m = threadIdx.x + u * NT;
        vx[u] = vp[u] = hh[u] = 0.0;
        if (m < N) {
            vx[u] = px[0];
            vp[u] = px[to_p];
            hh[u] = a.hann[m];
        }
        px += ahead;
    }
    if (scan_other)
        for (uint32_t m = threadIdx.x; m < N; m += NT) {
            const uint64_t sm = (uint64_t)a.from + m;
            nan_seen |= __builtin_isnan(a.hist[hat(a.lay, sm, co0, particle)] - mean_o0) ||
                        __builtin_isnan(a.hist[hat(a.lay, sm, co1, particle)] - mean_o1);
        }
#pragma unroll
    for (uint32_t u = 0; u < LP; ++u) {
        const uint32_t m = threadIdx.x + u * NT;
        if (m < N) {
            const double x = vx[u] - mean_x, xp = vp[u] - mean_p;
            nan_seen |= __builtin_isnan(x) || __builtin_isnan(xp);
            Cplx z{x * hh[u], xp * hh[u]};
            if constexpr (CZ) z = cmul(z, a.chirp[m]);
            buf[m] = z;
        }
    }
    if constexpr (CZ)
        for (uint32_t m = N + threadIdx.x; m < M; m += NT) buf[m] = Cplx{0.0, 0.0};
    if (__syncthreads_or(nan_seen)) {
        if (threadIdx.x == 0) *o = __builtin_nan("");
        return;
    }
    wh_fft<NT, PMAX>(buf, a.plan, a.tw, a.frag);
    if constexpr (CZ) {
        for (uint32_t k = threadIdx.x; k < M; k += NT) {
            const uint32_t l = k;
            const Cplx z = cmul(buf[l], a.bhat[k]);
            buf[l] = Cplx{z.re, -z.im};
        }
        __syncthreads();
        wh_fft<NT, PMAX>(buf, a.plan, a.tw, a.frag);
    }
    // first maximum of |X_k|, k < N: the largest square (one square root of it for
    // the workgroup instead of one an entry), then the lowest k whose root equals
    // its root; only squares within a few units of it can
    auto square = [&](uint32_t k) {
        const Cplx z = buf[k];
        return z.re * z.re + z.im * z.im;
    };
    double sq[LP], top = -1.0;
#pragma unroll
    for (uint32_t u = 0; u < LP; ++u) {
        const uint32_t k = threadIdx.x + u * NT;
        const double v = square(min(k, N - 1));
        sq[u] = k < N ? v : -1.0;
        top = sq[u] > top ? sq[u] : top;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double o2 = __shfl_xor(top, off);
        top = o2 > top ? o2 : top;
    }
    if (threadIdx.x == 0) first = 0xffffffffu;
    if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = top;
    __syncthreads();
    top = sv[threadIdx.x % (NT / 64)];
#pragma unroll
    for (int off = (int)NT / 128; off > 0; off >>= 1) {
        const double o2 = __shfl_xor(top, off);
        top = o2 > top ? o2 : top;
    }
    const double near = top * (1.0 - 0x1p-50), root = sqrt(top);
    uint32_t i = 0xffffffffu;
#pragma unroll
    for (int u = (int)LP - 1; u >= 0; --u)
        if (sq[u] >= near) {
            asm volatile("" : "+v"(sq[u]));  // no root ahead of the branch
            if (sqrt(sq[u]) == root) i = threadIdx.x + u * NT;
        }
    if (i != 0xffffffffu) atomicMin(&first, i);
    __syncthreads();
    if (threadIdx.x == 0) {
        auto mag = [&](uint32_t k) { return sqrt(square(k)); };
        // (a scan from entry 0 on never leaves one that is NaN, and passes later ones by)
        const bool at_zero = first == 0xffffffffu || __builtin_isnan(square(0));
        *o = interp_tune_at(mag, N, at_zero ? 0u : first, a.cos_n, a.sin_n);
    }
}

__global__ void k_mr_zero(uint32_t *__restrict__ p, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------- host plan
struct MrTables {
    uint32_t M = 0, N1 = 0, N2 = 0;  // M = 0: no plan for this length
    MrPlan p1{}, p2{};
    Cplx *tw1 = nullptr, *tw2 = nullptr, *twm = nullptr;
    Cplx *chirp = nullptr, *bhat = nullptr;  // chirp-z plans only
};

// Radix plan of a {2,3,5,7}-smooth length: radix 8 while it divides, then 4,
// 2, 3, 5, 7. False when L has another prime factor.
static bool radix_plan(uint32_t L, MrPlan &p)
{
    p = MrPlan{};
    p.L = L;
    uint32_t r = L;
    auto take = [&](uint32_t R) {
        while (r % R == 0 && p.n_pass < (uint32_t)kMrMaxPasses) {
            p.radices |= (uint64_t)R << (4 * p.n_pass++);
            r /= R;
        }
    };
    take(8); take(4); take(2); take(3); take(5); take(7);
    return r == 1;
}

// N = N1 x N2 with N1 <= N2 <= kMrPmax, N1 >= 2 and N1 as large as possible.
static bool split(uint32_t N, uint32_t &N1, uint32_t &N2)
{
    N1 = N2 = 0;
    for (uint32_t a = 2; (uint64_t)a * a <= N; ++a)
        if (N % a == 0 && N / a <= kMrPmax) { N1 = a; N2 = N / a; }
    return N1 != 0;
}

// Both factors of a split length have radix plans.
static bool plan_length(uint32_t M, MrTables &t)
{
    uint32_t r = M;
    for (uint32_t q : {2u, 3u, 5u, 7u})
        while (r % q == 0) r /= q;
    if (r != 1) return false;
    uint32_t N1, N2;
    if (!split(M, N1, N2) || !radix_plan(N1, t.p1) || !radix_plan(N2, t.p2)) return false;
    t.M = M; t.N1 = N1; t.N2 = N2;
    return true;
}

template <class T>
static T *upload(const std::vector<T> &v, hipStream_t s, const char *what)
{
    T *d = nullptr;
    hip_check(device_malloc(&d, v.size() * sizeof(T)), what);
    hip_check(hipMemcpyAsync(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s), "hipMemcpyAsync");
    return d;
}

using CplxL = std::complex<long double>;

// Forward DFT of a {2,3,5,7}-smooth length in long double (the chirp-z filter
// spectrum): recursive decimation in time by the smallest prime factor r of
// n = r m, X[k + m q] = sum_s W_n^{s (k + m q)} Y_s[k], Y_s the DFT of x[s + r j].
// root[e] = W_M^e; a sub-length n uses W_n^e = root[e M / n].
static void host_dft_rec(const CplxL *in, size_t stride, CplxL *out, size_t n, const std::vector<CplxL> &root,
                         size_t M, std::vector<CplxL> &tmp)
{
    if (n == 1) { out[0] = in[0]; return; }
    size_t r = 2;
    while (n % r) ++r;
    const size_t m = n / r, rs = M / n;
    for (size_t s = 0; s < r; ++s) host_dft_rec(in + s * stride, stride * r, out + s * m, m, root, M, tmp);
    CplxL *t = tmp.data();
    for (size_t k = 0; k < m; ++k)
        for (size_t q = 0; q < r; ++q) {
            const size_t kk = k + m * q;
            CplxL acc = out[k];
            for (size_t s = 1; s < r; ++s) acc += out[s * m + k] * root[((s * kk) % n) * rs];
            t[kk] = acc;
        }
    std::copy(t, t + n, out);
}

static std::vector<CplxL> host_dft(const std::vector<CplxL> &x)
{
    const size_t M = x.size();
    const long double two_pi = 6.283185307179586476925286766559005768L;
    std::vector<CplxL> root(M), out(M), tmp(M);
    for (size_t q = 0; q < M; ++q) {
        const long double ang = two_pi * (long double)q / (long double)M;
        root[q] = CplxL(cosl(ang), -sinl(ang));
    }
    host_dft_rec(x.data(), 1, out.data(), M, root, M, tmp);
    return out;
}

// Tables of one length (cached per device): the direct plan of a
// {2,3,5,7}-smooth N, else the chirp-z plan over the smallest smooth M >=
// 2N - 1 that splits; M = 0 when neither exists (M would exceed kMrPmax^2).
static const MrTables *mr_tables(uint32_t N, hipStream_t s)
{
    static std::mutex mu;
    static std::map<std::pair<int, uint32_t>, MrTables> cache;
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find({dev, N});
    if (it != cache.end()) return it->second.M ? &it->second : nullptr;
    MrTables t;
    bool cz = false;
    if (!plan_length(N, t)) {
        cz = true;
        const uint64_t lo = 2ull * N - 1, hi = (uint64_t)kMrPmax * kMrPmax;
        for (uint64_t M = lo; M <= hi; ++M)
            if (plan_length((uint32_t)M, t)) break;
        if (!t.M) {
            cache[{dev, N}] = MrTables{};
            return nullptr;
        }
    }
    const uint32_t M = t.M, N1 = t.N1, N2 = t.N2;
    const long double two_pi = 6.283185307179586476925286766559005768L, pi = two_pi / 2;
    auto roots = [&](uint32_t L) {
        std::vector<Cplx> v(L);
        for (uint32_t q = 0; q < L; ++q) {
            const long double ang = two_pi * (long double)q / (long double)L;
            v[q] = Cplx{(double)cosl(ang), (double)-sinl(ang)};
        }
        return v;
    };
    const std::vector<Cplx> r1 = roots(N1), r2 = roots(N2), rM = roots(M);
    // step twiddles W_M^{k1 n2}, reduced exactly mod M
    std::vector<Cplx> m((size_t)M);
    for (uint64_t k1 = 0; k1 < N1; ++k1)
        for (uint64_t n2 = 0; n2 < N2; ++n2) m[k1 * N2 + n2] = rM[(k1 * n2) % M];
    t.tw1 = upload(r1, s, "hipMalloc(mixed-radix twiddles)");
    t.tw2 = upload(r2, s, "hipMalloc(mixed-radix twiddles)");
    t.twm = upload(m, s, "hipMalloc(mixed-radix step twiddles)");
    if (cz) {
        // chirp c_m = exp(-i pi (m^2 mod 2N) / N) (m^2 exact in 64 bits), filter
        // b_j = conj(c_j) for |j| < N (j mod M), B = DFT_M(b) stored [k1][k2]
        std::vector<Cplx> chirp(N), bhat((size_t)M);
        std::vector<CplxL> b((size_t)M, CplxL(0, 0));
        for (uint64_t q = 0; q < N; ++q) {
            const long double ang = pi * (long double)((q * q) % (2ull * N)) / (long double)N;
            const long double c = cosl(ang), sn = sinl(ang);
            chirp[q] = Cplx{(double)c, (double)-sn};
            b[q] = CplxL(c, sn);
            if (q > 0) b[M - q] = b[q];
        }
        const std::vector<CplxL> B = host_dft(b);
        for (size_t k1 = 0; k1 < N1; ++k1)
            for (size_t k2 = 0; k2 < N2; ++k2) {
                const CplxL z = B[k1 + (size_t)N1 * k2];
                bhat[k1 * N2 + k2] = Cplx{(double)z.real(), (double)z.imag()};
            }
        t.chirp = upload(chirp, s, "hipMalloc(chirp)");
        t.bhat = upload(bhat, s, "hipMalloc(chirp-z filter)");
    }
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
    cache[{dev, N}] = t;
    return &cache[{dev, N}];
}

static uint64_t mr_budget()
{
    const char *e = std::getenv("HM_FFT_ROW_BYTES");
    if (e && *e) {
        const unsigned long long v = std::strtoull(e, nullptr, 10);
        if (v > 0) return v;
    }
    return 8ull << 30;  // a few percent of the device memory: large batches, few launches
}

// largest divisor of v that is at most cap
static uint32_t divisor_at_most(uint32_t v, uint32_t cap)
{
    for (uint32_t d = std::min(v, cap); d > 1; --d)
        if (v % d == 0) return d;
    return 1;
}

template <class K>
static void set_lds(K kernel, size_t bytes)
{
    hip_check(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes),
              "hipFuncSetAttribute");
}

// ---------------------------------------------------------------- whole-signal plans
// Passes of the direct transform of L: primes from 17 up to kWhPrimeMax by one
// pass each, the rest by as few passes as the radices 2 .. 13 and 16 allow (each
// pass is a trip through LDS behind two barriers, 4000 to 7000 cycles of a
// workgroup of 1024 threads at 10^4 points whatever its radix), of the fewest the
// one with the smallest sum of radices; grouped as wh_fft runs them. `gen` = the
// sum of the primes (their passes cost about 2R operations per point against a
// few tens for a small radix).
static uint32_t udiv_magic(uint32_t d) { return d == 1 ? 0u : (uint32_t)((1ull << 32) / d + 1); }

constexpr uint32_t kSmallRadices[] = {16, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// The best list of radices (not increasing, from entry `from` on) with product r:
// the fewest; then one with a radix whose stores of the first pass share banks
// least (stride R entries of 16 bytes); then the smallest sum.
static bool few_radices(uint32_t r, size_t from, std::vector<uint32_t> &best)
{
    best.clear();
    if (r == 1) return true;
    auto cost = [](const std::vector<uint32_t> &v) {
        uint32_t sum = 0, shared = 8;
        for (uint32_t R : v) {
            sum += R;
            shared = std::min(shared, R & (0u - R));
        }
        return (uint64_t)v.size() << 32 | shared << 16 | sum;
    };
    bool found = false;
    for (size_t q = from; q < std::size(kSmallRadices); ++q) {
        std::vector<uint32_t> rest;
        if (r % kSmallRadices[q] || !few_radices(r / kSmallRadices[q], q, rest)) continue;
        rest.push_back(kSmallRadices[q]);
        if (!found || cost(rest) < cost(best)) best = rest;
        found = true;
    }
    return found;
}

static bool wh_radix_plan(uint32_t L, WhPlan &p, uint32_t &gen)
{
    p = WhPlan{};
    p.L = L;
    gen = 0;
    uint32_t r = L, Ns = 1, tw = 0;
    auto push = [&](uint32_t R) {
        if (p.n_pass == (uint32_t)kWhMaxPasses) return false;
        WhPass &q = p.pass[p.n_pass++];
        q.R = R; q.Ns = Ns; q.B = L / R;
        q.m_ns = udiv_magic(Ns); q.m_b = udiv_magic(q.B); q.m_h1 = udiv_magic((R - 1) / 2 + 1);
        q.frag = kNoFrag;
        q.tw = tw;
        if (Ns > 1) tw += R > 16 ? (R - 1) * Ns : Ns;
        q.root = tw;
        if (R > 16) tw += (R - 1) / 2 + 1;
        Ns *= R;
        return true;
    };
    std::vector<uint32_t> primes, small;
    uint32_t smooth = 1;
    for (uint32_t q : {2u, 3u, 5u, 7u, 11u, 13u})
        for (; r % q == 0; r /= q) smooth *= q;
    for (uint32_t q = 17; r > 1 && q <= kWhPrimeMax; q += 2)
        for (; r % q == 0; r /= q) {
            primes.push_back(q);
            gen += q;
        }
    if (r != 1 || !few_radices(smooth, 0, small)) return false;
    for (uint32_t R : {3u, 5u, 7u, 9u, 11u, 13u, 0u, 6u, 10u, 2u, 12u, 4u, 8u, 16u}) {
        for (uint32_t v : R ? small : primes)
            if ((!R || v == R) && !push(v)) return false;
    }
    return true;
}

struct WhTables {
    bool ok = false, cz = false;
    uint32_t M = 0, nt = 0;
    WhPlan plan{};
    Cplx *tw = nullptr, *chirp = nullptr, *bhat = nullptr, *frag = nullptr;
};

static uint32_t wh_threads(uint32_t M)
{
    uint32_t nt = 64;
    while (nt * kWhPoints < M) nt *= 2;
    return nt;
}

// A prime pass runs on the matrix cores where its tiles fit the registers of the
// plan's wavefronts; others (17, 19 and 37 near the most points of a shape, 257,
// primes above 64 in the shapes of one and two wavefronts) take their sums on the
// vector units. ns per signal with and without, at 2e8 points in all: 437 points (19 x 23) 4.9 and 6.2, 2491 (47 x 53) 28
// and 40, 4087 (61 x 67) 58 and 99, 10001 (73 x 137) 184 and 331.
static bool matrix_pass(const WhPass &ps, uint32_t nt)
{
    return ps.R > 16 && matrix_tiles(ps.R, ps.B) <= kMatrixRounds * (nt / 64);
}

// Whether N's own transform beats chirp-z over more than twice the points: without
// prime passes always; with them while their sum is at most kWhCzGen or all run
// on the matrix cores, over enough butterflies to fill a pass (a wavefront's worth
// of a matrix tile's 16; a matrix pass of few rows always). ns per signal, direct
// and chirp-z: 323 points (17 x 19) 4.4 and 8.0, 1207 (17 x 71) 18 and 23, 2010
// (30 x 67) 23 and 47, 2869 (19 x 151) 58 and 90; but 67 points 5.7 and 3.5, 501
// (3 x 167) 12.8 and 10.7, 755 (5 x 151) 23 and 18, 1799 (7 x 257) 63 and 48.
constexpr uint32_t kWhCzGen = 128;
static bool prefer_direct(const WhPlan &p, uint32_t gen)
{
    const uint32_t nt = wh_threads(p.L);
    bool all_matrix = true, filled = true;
    for (uint32_t q = 0; q < p.n_pass; ++q) {
        const WhPass &ps = p.pass[q];
        if (ps.R <= 16) continue;
        const bool m = matrix_pass(ps, nt);
        all_matrix &= m;
        filled &= ps.B >= 16 || (m && gen <= kWhCzGen);
    }
    return filled && (gen <= kWhCzGen || all_matrix);
}

// The time of chirp-z over a plan's points, in about 5e-5 ns. A pass takes its
// butterflies a wavefront of 64 at a time, whole or not, at 18 to 26 units a point by its
// radix; a point takes 120 beside the passes (samples, filter, maximum), more in a small
// length whose radices are all multiples of 4, which share banks; a thread takes 400 and
// 60 a pass (start, barriers). Half as much again where one workgroup of 512 threads
// leaves no room on the CU for a second. ns per signal: 1779 points over 4096 = 16^3 46.3,
// over 3564 = 4 x 9 x 9 x 11 44.2, over 3584 = 7 x 8 x 8 x 8 40.3; 281 over 560 = 7 x 8 x 10
// 4.9, over 567 = 7 x 9 x 9 (63 butterflies of radix 9) 4.3; 2520 over 5120 87, over 5040 58.
static uint64_t chirp_cost(const WhPlan &p, bool alone)
{
    static constexpr uint32_t per_point[17] = {0, 0, 26, 26, 24, 20, 18, 20, 19, 20, 19, 24, 18, 26, 0, 0, 22};
    uint64_t c = (400ull + 60 * p.n_pass) * wh_threads(p.L) + 120ull * p.L;
    uint32_t shared = 8;
    for (uint32_t q = 0; q < p.n_pass; ++q) {
        const WhPass &ps = p.pass[q];
        c += (uint64_t)per_point[ps.R] * ps.R * ((ps.B + 63) / 64 * 64);
        shared = std::min(shared, ps.R & (0u - ps.R));
    }
    if (p.L <= 256 * kWhPoints) c += (shared == 8 ? 80ull : shared == 4 ? 12ull : 0ull) * p.L;
    return alone ? c + c / 2 : c;
}

// Whole-signal plan of a window length (cached per device): the direct transform
// or chirp-z over a smooth M >= 2N - 1 that fits, by the rule above; the direct
// transform also where no chirp-z length fits; none when N does not fit or has a
// prime above kWhPrimeMax and no chirp-z length fits. M is the one of the least cost:
// 501 points take 1008 = 7 x 12 x 12.
static const WhTables *wh_tables(uint32_t N, hipStream_t s)
{
    static std::mutex mu;
    static std::map<std::pair<int, uint32_t>, WhTables> cache;
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find({dev, N});
    if (it != cache.end()) return it->second.ok ? &it->second : nullptr;
    int v = 0;
    hip_check(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev), "hipDeviceGetAttribute");
    // the kernels' own LDS (reductions) comes on top of the signal
    size_t fixed = 0;
    for (const void *k : {(const void *)k_wh_tune<false, kWhThreads>, (const void *)k_wh_tune<true, kWhThreads>}) {
        hipFuncAttributes fa{};
        hip_check(hipFuncGetAttributes(&fa, k), "hipFuncGetAttributes");
        fixed = std::max(fixed, (size_t)fa.sharedSizeBytes);
    }
    const size_t lds = (size_t)v > fixed ? (size_t)v - fixed : 0;
    auto fits = [&](uint32_t M) { return M <= kWhPmax && (size_t)M * sizeof(Cplx) <= lds; };
    WhTables t;
    WhPlan pd{};
    uint32_t gen = 0;
    const bool direct = fits(N) && wh_radix_plan(N, pd, gen);
    uint32_t Mcz = 0;
    WhPlan pc{};
    const bool own = direct && prefer_direct(pd, gen);
    if (!own) {
        hipFuncAttributes fa512{};
        hip_check(hipFuncGetAttributes(&fa512, (const void *)k_wh_tune<true, 512>), "hipFuncGetAttributes");
        uint64_t cost = ~0ull;
        for (uint64_t M = 2ull * N - 1; M <= 4ull * N && M <= kWhPmax && fits((uint32_t)M); ++M) {
            uint32_t g = 0;
            WhPlan pm{};
            if (!wh_radix_plan((uint32_t)M, pm, g) || g) continue;
            const bool alone = wh_threads((uint32_t)M) == 512 && 2 * (M * sizeof(Cplx) + fa512.sharedSizeBytes) > (size_t)v;
            const uint64_t c = chirp_cost(pm, alone);
            if (c >= cost) continue;
            cost = c;
            Mcz = (uint32_t)M;
            pc = pm;
        }
    }
    if (own || (direct && !Mcz)) {
        t.ok = true; t.cz = false; t.M = N; t.plan = pd;
    } else if (Mcz) {
        t.ok = true; t.cz = true; t.M = Mcz; t.plan = pc;
    }
    if (!t.ok) {
        cache[{dev, N}] = WhTables{};
        return nullptr;
    }
    const uint32_t M = t.M;
    t.nt = wh_threads(M);
    const long double two_pi = 6.283185307179586476925286766559005768L, pi = two_pi / 2;
    std::vector<Cplx> w;
    auto root = [&](uint64_t num, uint64_t den) {
        const long double ang = two_pi * (long double)(num % den) / (long double)den;
        w.push_back(Cplx{(double)cosl(ang), (double)-sinl(ang)});
    };
    for (uint32_t p = 0; p < t.plan.n_pass; ++p) {
        const WhPass &ps = t.plan.pass[p];
        if (ps.Ns > 1)
            for (uint32_t r = 1; r < (ps.R > 16 ? ps.R : 2u); ++r)
                for (uint32_t k = 0; k < ps.Ns; ++k) root((uint64_t)k * r, (uint64_t)ps.Ns * ps.R);
        if (ps.R > 16)
            for (uint32_t q = 0; q <= (ps.R - 1) / 2; ++q) root(q, ps.R);
    }
    if (w.empty()) w.push_back(Cplx{1.0, 0.0});
    t.tw = upload(w, s, "hipMalloc(whole-signal twiddles)");
    // Root matrices in the lanes' order of the matrix instruction: lane l of step t
    // of row tile i holds row q = 16 i + l % 16, column r = 4 t + l / 16 + 1 (zero beyond H).
    std::vector<Cplx> frag;
    for (uint32_t p = 0; p < t.plan.n_pass; ++p) {
        WhPass &ps = t.plan.pass[p];
        if (!matrix_pass(ps, t.nt)) continue;
        ps.frag = (uint32_t)frag.size();
        const uint32_t H = (ps.R - 1) / 2;
        for (uint32_t i = 0; i < matrix_rows(ps.R); ++i)
            for (uint32_t st = 0; st < matrix_steps(ps.R); ++st)
                for (uint32_t l = 0; l < 64; ++l) {
                    const uint32_t q = 16 * i + l % 16, r = 4 * st + l / 16 + 1;
                    const long double ang = two_pi * (long double)(q * r % ps.R) / (long double)ps.R;
                    frag.push_back(q <= H && r <= H ? Cplx{(double)cosl(ang), (double)sinl(ang)} : Cplx{0.0, 0.0});
                }
    }
    if (!frag.empty()) t.frag = upload(frag, s, "hipMalloc(whole-signal root matrices)");
    if (t.cz) {
        // chirp c_m = exp(-i pi (m^2 mod 2N) / N), filter b_j = conj(c_j) for
        // |j| < N (j mod M), B = DFT_M(b) in natural order
        std::vector<Cplx> chirp(N), bhat(M);
        std::vector<CplxL> b(M, CplxL(0, 0));
        for (uint64_t q = 0; q < N; ++q) {
            const long double ang = pi * (long double)((q * q) % (2ull * N)) / (long double)N;
            const long double c = cosl(ang), sn = sinl(ang);
            chirp[q] = Cplx{(double)c, (double)-sn};
            b[q] = CplxL(c, sn);
            if (q > 0) b[M - q] = b[q];
        }
        const std::vector<CplxL> B = host_dft(b);
        for (uint32_t k = 0; k < M; ++k) bhat[k] = Cplx{(double)B[k].real(), (double)B[k].imag()};
        t.chirp = upload(chirp, s, "hipMalloc(chirp)");
        t.bhat = upload(bhat, s, "hipMalloc(chirp-z filter)");
    }
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
    cache[{dev, N}] = t;
    return &cache[{dev, N}];
}

template <bool CZ, uint32_t NT>
static void launch_wh(const WhArgs &a0, uint32_t nt, uint32_t n, size_t lds_bytes, hipStream_t s)
{
    if constexpr (NT > 64)
        if (nt < NT) return launch_wh<CZ, NT / 2>(a0, nt, n, lds_bytes, s);
    auto k = k_wh_tune<CZ, NT>;
    set_lds(k, lds_bytes);
    WhArgs a = a0;
    // 2 signals per particle, one workgroup each: grids below 2^31 workgroups
    const uint32_t chunk = 1u << 29;
    for (uint32_t p0 = 0; p0 < n; p0 += chunk) {
        const uint32_t nb = std::min(chunk, n - p0);
        a.p0 = p0;
        hipLaunchKernelGGL(k, dim3(2 * nb), dim3(NT), lds_bytes, s, a);
        launch_check("k_wh_tune");
    }
}

// The whole-signal transform of one window; false (nothing launched) when the
// length has no whole-signal plan.
static bool fft_tune_whole(const double *hist, HistLayout lay, uint32_t n, const double *means, uint32_t from,
                           uint32_t N, const double *hann, double *out, uint32_t window, hipStream_t s)
{
    const WhTables *t = wh_tables(N, s);
    if (!t) return false;
    if (n == 0) return true;
    WhArgs a{};
    a.hist = hist; a.lay = lay; a.means = means; a.n = n; a.from = from; a.N = N; a.M = t->M;
    a.plan = t->plan; a.hann = hann; a.tw = t->tw;
    a.cos_n = std::cos(2.0 * M_PI / (double)N); a.sin_n = std::sin(2.0 * M_PI / (double)N);
    a.frag = t->frag; a.chirp = t->chirp; a.bhat = t->bhat;
    a.out = out; a.window = window;
    const size_t lds_bytes = (size_t)t->M * sizeof(Cplx);
    LaunchTimer timer("k_wh_tune", s);
    if (t->cz) launch_wh<true, kWhThreads>(a, t->nt, n, lds_bytes, s);
    else launch_wh<false, kWhThreads>(a, t->nt, n, lds_bytes, s);
    return true;
}

bool fft_tune_mixed(const double *hist, HistLayout lay, uint32_t n, const double *means, uint32_t from, uint32_t N,
                    const double *hann, double *out, uint32_t window, hipStream_t s)
{
    if (N < 2) return false;
    if (fft_tune_whole(hist, lay, n, means, from, N, hann, out, window, s)) return true;
    const MrTables *t = mr_tables(N, s);
    if (!t) return false;
    if (n == 0) return true;
    const bool cz = t->chirp != nullptr;
    MrArgs a{};
    a.hist = hist; a.lay = lay; a.means = means; a.n = n; a.from = from; a.N = N; a.M = t->M;
    a.N1 = t->N1; a.N2 = t->N2; a.p1 = t->p1; a.p2 = t->p2;
    a.C = divisor_at_most(a.N2, kMrPmax / a.N1);
    a.RR = divisor_at_most(a.N1, kMrPmax / a.N2);
    a.hann = hann; a.tw1 = t->tw1; a.tw2 = t->tw2; a.twm = t->twm; a.chirp = t->chirp; a.bhat = t->bhat;
    a.out = out; a.window = window;
    const size_t lds_cols = (size_t)a.C * lds_len_odd(a.N1) * sizeof(Cplx);
    const size_t lds_rows = (size_t)a.RR * lds_len(a.N2) * sizeof(Cplx);
    // scratch per particle (both planes): the M-point work arrays, magnitudes, flags
    const uint64_t per_particle = 2 * ((uint64_t)sizeof(Cplx) * a.M + 8ull * N) + 8;
    // every grid below 2^31 threads: 2 signals per particle, up to per_sig
    // workgroups of kMrThreads per signal
    const uint64_t per_sig = std::max<uint64_t>({1, a.N2 / a.C, a.N1 / a.RR});
    const uint64_t max_batch = ((1ull << 31) / kMrThreads) / (2 * per_sig);
    const uint32_t batch =
        (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({(uint64_t)n, mr_budget() / per_particle, max_batch}));
    const size_t nsig_max = 2 * (size_t)batch;
    const size_t y_bytes = nsig_max * (size_t)a.M * sizeof(Cplx), mag_bytes = nsig_max * (size_t)N * 8;
    char *ws = static_cast<char *>(workspace(y_bytes + mag_bytes + nsig_max * 4 + 256, 3));
    a.Y = reinterpret_cast<Cplx *>(ws);
    a.mags = reinterpret_cast<double *>(ws + y_bytes);
    a.flags = reinterpret_cast<uint32_t *>(ws + y_bytes + mag_bytes);
    if (cz) {
        set_lds(k_mr_columns<true>, lds_cols);
        set_lds(k_mr_rows<true>, lds_rows);
        set_lds(k_mr_final, lds_cols);
    } else {
        set_lds(k_mr_columns<false>, lds_cols);
        set_lds(k_mr_rows<false>, lds_rows);
    }
    for (uint32_t p0 = 0; p0 < n; p0 += batch) {
        const uint32_t nb = std::min(batch, n - p0);
        a.p0 = p0;
        a.nsig = 2 * nb;
        hipLaunchKernelGGL(k_mr_zero, dim3((a.nsig + 255) / 256), dim3(256), 0, s, a.flags, a.nsig);
        launch_check("k_mr_zero");
        // grids of 8 x (workgroups per XCD); see mr_virtual
        const uint32_t cols = a.nsig * (a.N2 / a.C), rows = a.nsig * (a.N1 / a.RR);
        const dim3 gc((cols + 7) / 8 * 8), gr((rows + 7) / 8 * 8);
        {
            LaunchTimer timer("k_mr_columns", s);
            if (cz) hipLaunchKernelGGL(k_mr_columns<true>, gc, dim3(kMrThreads), lds_cols, s, a);
            else hipLaunchKernelGGL(k_mr_columns<false>, gc, dim3(kMrThreads), lds_cols, s, a);
            launch_check("k_mr_columns");
        }
        {
            LaunchTimer timer("k_mr_rows", s);
            if (cz) hipLaunchKernelGGL(k_mr_rows<true>, gr, dim3(kMrThreads), lds_rows, s, a);
            else hipLaunchKernelGGL(k_mr_rows<false>, gr, dim3(kMrThreads), lds_rows, s, a);
            launch_check("k_mr_rows");
        }
        if (cz) {
            LaunchTimer timer("k_mr_final", s);
            hipLaunchKernelGGL(k_mr_final, gc, dim3(kMrThreads), lds_cols, s, a);
            launch_check("k_mr_final");
        }
        LaunchTimer timer("k_mr_tune", s);
        if (cz) hipLaunchKernelGGL(k_mr_tune<true>, dim3(a.nsig), dim3(kMrThreads), 0, s, a);
        else hipLaunchKernelGGL(k_mr_tune<false>, dim3(a.nsig), dim3(kMrThreads), 0, s, a);
        launch_check("k_mr_tune");
    }
    return true;
}

}  // namespace hm
