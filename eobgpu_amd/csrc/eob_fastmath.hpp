// Logarithm, division, square and cube roots for the integrator's right-hand side.
//
// The right-hand side runs as one wavefront per binary, so its cost is the
// length of its instruction stream.  The device library's log carries a
// double-double evaluation (about 90 instructions besides its constants); the
// version here uses the textbook reduction and series (about 45), with every
// multiply-add written as fma() and contraction of the rest switched off, so
// that a host build rounds exactly as the device build does; within 1 ulp.
//
// log_pos: x = m 2^e with m in [sqrt(1/2), sqrt(2)); with f = m - 1 and
//   s = f / (2 + f), log(1 + f) = 2 atanh(s) = 2s + s R(s^2),
//   R(z) = sum_{k>=1} 2 z^k / (2k + 1), rearranged as
//   f - (f^2/2 - s (f^2/2 + R)) so that the exact f leads (the arrangement of
//   fdlibm's e_log.c).  |s| <= 0.1716, z <= 0.0295.  R is a polynomial of
//   degree 7 obtained by Chebyshev economization (Lanczos) of the series of
//   R(z)/z on [0, 0.0295]: the series to z^40 in exact rationals, rewritten
//   in Chebyshev polynomials of t = 2z/0.0295 - 1, cut after T_6 and rewritten
//   in powers of z; with the coefficients rounded to double, |R - poly| is
//   below 8.4e-18 on the interval (the Taylor series needs degree 10 for
//   that), which moves log by under 0.02 ulp (log_series_coefficients.py
//   derives and checks them).
// ln 2 is split into a 31-bit head (e ln2_hi is exact for |e| < 2^22) and the
// rounded remainder.
#pragma once
#include <cmath>

#ifndef EOB_HD
#ifdef __HIPCC__
#define EOB_HD __host__ __device__ __forceinline__
#else
#define EOB_HD inline   // host-only build (the unit test's probe)
#endif
#endif

namespace eob {

constexpr double kLn2Hi = 0x1.62e42fec00000p-1;       // ln 2 with the low 22 mantissa bits cleared
constexpr double kLn2Lo = 0x1.d1cf79abc9e3bp-32;      // ln 2 - kLn2Hi, rounded
constexpr double kSqrtHalf = 0x1.6a09e667f3bcdp-1;    // sqrt(1/2)

// a / b and 1 / b for normal, finite operands with a normal result: the
// hardware reciprocal estimate refined by two Newton steps, then one residual
// correction (Markstein's method).  The quotient rounds as IEEE division on
// such operands; the library's division adds scaling steps for the extreme
// exponent ranges that these arguments never reach.  Other types divide.
// A host build (the unit test) starts from the reciprocal rounded to single
// precision, a coarser estimate than the hardware's, so that it exercises
// the refinement.
EOB_HD double rcp_estimate(double b) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcp(b);
#else
    return (double)(float)(1.0 / b);
#endif
}
EOB_HD double refined_rcp(double b) {
    double y = rcp_estimate(b);
    y = fma(y, fma(-b, y, 1.0), y);
    y = fma(y, fma(-b, y, 1.0), y);
    return y;
}
template <class T>
EOB_HD T qdiv(T a, T b) { return a / b; }
template <class T>
EOB_HD T qrcp(T b) { return 1.0 / b; }
EOB_HD double qdiv(double a, double b) {
    const double y = refined_rcp(b);
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}
EOB_HD double qrcp(double b) {
    const double y = refined_rcp(b);
    return fma(fma(-b, y, 1.0), y, y);
}

// natural log of a positive finite x, within 1 ulp; NaN for every other x
// (0, negative, infinite or NaN), which the integrator treats as a failed binary
EOB_HD double log_pos(double x) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    int e;
    double m = frexp(x, &e);   // x = m 2^e, m in [1/2, 1)
    const bool lo = m < kSqrtHalf;
    m = lo ? m + m : m;
    e = lo ? e - 1 : e;
    const double f = m - 1.0;   // exact
    const double s = qdiv(f, 2.0 + f);
    const double z = s * s;
    double R = 0x1.2b6ada4e6cac0p-3;   // R(z)/z to degree 6, economized (see above)
    R = fma(R, z, 0x1.39fcd91739d16p-3);
    R = fma(R, z, 0x1.7462c0aff40b1p-3);
    R = fma(R, z, 0x1.c71c62ba3869bp-3);
    R = fma(R, z, 0x1.2492492e143e6p-2);
    R = fma(R, z, 0x1.999999999519ap-2);
    R = fma(R, z, 0x1.5555555555558p-1);
    const double hfsq = (0.5 * f) * f;
    const double dk = (double)e;
    const double t = fma(s, fma(R, z, hfsq), dk * kLn2Lo);
    const double res = fma(dk, kLn2Hi, -((hfsq - t) - f));
    return (x > 0.0 && x < HUGE_VAL) ? res : NAN;
}

// sqrt(x) for positive normal x: the hardware reciprocal-square-root
// estimate y, then Goldschmidt's iteration (g = x y, h = y/2; one step on the
// pair, two residual corrections on g) — correctly rounded in 20 000 of
// 20 000 simulated cases; the library's version adds range scaling and
// special-case selects these arguments never need.  Other types use sqrt.
EOB_HD double rsqrt_estimate(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rsq(x);
#else
    return (double)(float)(1.0 / sqrt(x));   // host build: a single-precision start, as for rcp_estimate
#endif
}
template <class T>
EOB_HD T qsqrt(T x) { return sqrt(x); }
EOB_HD double qsqrt(double x) {
    const double y = rsqrt_estimate(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    return g;
}

// sqrt(x) and 1/sqrt(x) together: the square root as qsqrt, and 2h (which
// Goldschmidt's iteration carries as 1/sqrt(x) to about 2^-44) refined by one
// Newton step for 1/g, within 1 ulp -- two fused multiply-adds instead of a
// separate reciprocal.
template <class T>
EOB_HD void qsqrt_recip(T x, T& root, T& inv) {
    root = sqrt(x);
    inv = 1.0 / root;
}
EOB_HD void qsqrt_recip(double x, double& root, double& inv) {
    const double y = rsqrt_estimate(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    g = fma(fma(-g, g, x), h, g);
    const double y2 = h + h;
    root = g;
    inv = fma(y2, fma(-g, y2, 1.0), y2);
}

// cube root of a positive normal x: a single-precision estimate of x^(-1/3)
// (hardware log2 and exp2), two Newton steps for z = x^(-1/3) (z += z (1 - x
// z^3) / 3, no division), y = x z^2 and one residual correction
// y += (x - y^3) z^2 / 3.  Within 1 ulp (0.71 in 20 000 simulated cases),
// about 23 instructions against 34 for the library's; NaN for 0 and NaN (and,
// on the device, for x < 0, whose log2 is NaN).
EOB_HD float rcbrt_estimate(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)x) * (-1.0f / 3.0f));
#else
    return (float)(1.0 / cbrt(x));   // host build: a single-precision start, as for rcp_estimate
#endif
}
EOB_HD double cbrt_pos(double x) {
    constexpr double kThird = 1.0 / 3.0;
    double z = (double)rcbrt_estimate(x);
    z = fma(z * kThird, fma(-x, (z * z) * z, 1.0), z);
    z = fma(z * kThird, fma(-x, (z * z) * z, 1.0), z);
    const double z2 = z * z;
    const double y = x * z2;
    return fma(fma(-(y * y), y, x) * kThird, z2, y);
}

EOB_HD unsigned long long double_bits(double v) {
    union {
        double d;
        unsigned long long u;
    } q{v};
    return q.u;
}

// x mod pi/2 for finite |x| >= 2^49 (Payne and Hanek's reduction): x = M 2^e with a
// 53-bit M, and the 128 bits of M (2^e / (2 pi) mod 1) below the point from the 192
// bits of 1/(2 pi) that meet them; returns the nearest quarter turn, the rest is
// r + w.
EOB_HD int reduce_huge(double x, double& r, double& w) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    constexpr unsigned long long kTurn[21] = {   // 1/(2 pi), 64 bits a word, from 2^64 down
        0ull, 0x28be60db9391054aull, 0x7f09d5f47d4d3770ull, 0x36d8a5664f10e410ull, 0x7f9458eaf7aef158ull, 0x6dc91b8e909374b8ull,
        0x01924bba82746487ull, 0x3f877ac72c4a69cfull, 0xba208d7d4baed121ull, 0x3a671c09ad17df90ull, 0x4e64758e60d4ce7dull,
        0x272117e2ef7e4a0eull, 0xc7fe25fff7816603ull, 0xfbcbc462d6829b47ull, 0xdb4d9fb3c9f2c26dull, 0xd3d18fd9a797fa8bull,
        0x5d49eeb1faf97c5eull, 0xcf41ce7de294a4baull, 0x9afed7ec47e35742ull, 0x1580cc11bf1edaeaull, 0xfc33ef0826bd0d87ull};
    constexpr double kRadHi = 0x1.921fb54442d18p-62, kRadLo = 0x1.1a62633145c07p-116;   // 2 pi 2^-64
    const auto high = [](unsigned long long a, unsigned long long b) {
#ifdef __HIP_DEVICE_COMPILE__
        return __umul64hi(a, b);
#else
        return (unsigned long long)(((unsigned __int128)a * b) >> 64);
#endif
    };
    const unsigned long long u = double_bits(fabs(x)), M = (u & 0xfffffffffffffull) | 0x10000000000000ull;
    const int o = (int)(u >> 52) - 1075 + 64, j = o >> 6, sh = o & 63;   // o >= 61; 1036 for infinities
    // M times words j + 2, j + 1 and j of the shifted bits, the carries upwards
    unsigned long long f0 = 0, f1 = 0, up = 0;
#pragma unroll 1
    for (int k = j + 2; k >= j; --k) {
        const unsigned long long t = sh ? (kTurn[k] << sh) | (kTurn[k + 1] >> (64 - sh)) : kTurn[k], lo = M * t;
        f1 = f0;
        f0 = lo + up;
        up = high(M, t) + (f0 < lo ? 1 : 0);
    }
    const unsigned long long q = (f0 + (1ull << 61)) >> 62;   // quarter turns, to nearest
    const long long g = (long long)(f0 - (q << 62));
    const double d0 = (double)g, d1 = (double)(g - (long long)d0) + (double)f1 * 0x1p-64;
    const double h = d0 * kRadHi, l = fma(d0, kRadHi, -h) + fma(d0, kRadLo, d1 * kRadHi);
    r = h + l;
    w = l - (r - h);
    if (fabs(x) > 0x1.fffffffffffffp1023) r = x - x;   // NaN
    if (x >= 0.0) return (int)q;
    r = -r;
    w = -w;
    return -(int)q;
}

// sin and cos of r + w + k pi/2, |r| <= 0.87: the Taylor series through r^17 and r^16
// (first omitted terms below 1e-18 of the result), w to first order.
EOB_HD void sincos_reduced(int k, double r, double w, double& s, double& c) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    const double z = r * r;
    double p = fma(z, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
    p = fma(p, z, 1.0 / 6227020800.0);
    p = fma(p, z, -1.0 / 39916800.0);
    p = fma(p, z, 1.0 / 362880.0);
    p = fma(p, z, -1.0 / 5040.0);
    p = fma(p, z, 1.0 / 120.0);
    p = fma(p, z, -1.0 / 6.0);
    double q = fma(z, 1.0 / 20922789888000.0, -1.0 / 87178291200.0);
    q = fma(q, z, 1.0 / 479001600.0);
    q = fma(q, z, -1.0 / 3628800.0);
    q = fma(q, z, 1.0 / 40320.0);
    q = fma(q, z, -1.0 / 720.0);
    q = fma(q, z, 1.0 / 24.0);
    const double v = fma(-0.5, z, 1.0);
    const double sr = r + fma(r * z, p, w * v);
    const double cr = v + fma(z * z, q, fma(-r, w, fma(-0.5, z, 1.0 - v)));
    const double a = (k & 1) ? cr : sr, b = (k & 1) ? sr : cr;
    s = (k & 2) ? -a : a;
    c = ((k + 1) & 2) ? -b : b;
}

// sin and cos of x (NaN for NaN) and true; but for |x| >= 2^49 false, and they are not set
// to anything useful.  r + w = x - n pi/2, where the first difference is exact and w is what the
// rounding of r leaves.  Within 9e-17 absolute, as the device library (8.7e-17; rms
// 2.8e-17 both).
EOB_HD bool sincos_bounded(double x, double& s, double& c) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    constexpr double kTwoOverPi = 0x1.45f306dc9c883p-1, kPio2Hi = 0x1.921fb54442d18p+0, kPio2Lo = 0x1.1a62633145c07p-54;
    constexpr double kInts = 0x1.8p52;   // added to: rounds to an integer, which the low word then holds
    const double m = fma(x, kTwoOverPi, kInts), n = m - kInts;
    const double t = fma(-n, kPio2Hi, x), r = fma(-n, kPio2Lo, t), w = fma(-n, kPio2Lo, t - r);
    sincos_reduced((int)(unsigned)double_bits(m), r, w, s, c);
    return !(fabs(x) >= 0x1p49);
}

// the same for every x (NaN for infinities)
EOB_HD void sincos_phase(double x, double& s, double& c) {
    if (sincos_bounded(x, s, c)) return;
    double r, w;
    const int k = reduce_huge(x, r, w);
    sincos_reduced(k, r, w, s, c);
}

}  // namespace eob
