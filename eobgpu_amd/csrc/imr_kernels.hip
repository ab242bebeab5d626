// Merger-ringdown attachment of the modes on the device: the NQC solve, the
// remnant and its QNMs, the ringdown coefficients and the template on the
// uniform grid with the NQC factor applied up to the attachment sample and the
// ringdown after it.
//
// Reference: SEOBNRv4PHM.compute_full_waveform (eob/seobnrv4phm.py:2308-2556),
// EOBCalculateNQCCoefficientsV4_freeattach (:1465-1683), EOBNonQCCorrection
// (:1686-1700), compute_MR_mode_free (:1779-1844), the fits of
// eob/eobstuff.py and the template sum of BBHWaveformTD (:720).
//
// Layout.  The splines of the modes are the batch's mode splines (coef
// [n][max_step][4 (2 nm + 1)]: Re and Im of h_j e^{i m_j phi}, then phi) and a
// second set of r and pr (rp [n][max_step][8]).  The attachment needs the
// modes only around two times per (binary, mode): the NQC time and the
// ringdown match time.  Each is a not-a-knot spline over the uniform-grid
// samples from a fixed start to the series' end; here the end is cut
// kImrAfter rows past the evaluation interval (the end condition's influence
// on that interval falls as 0.268 per row, 5e-18 at 31 rows), so one
// wavefront samples a whole window, one sample per lane, in one pass.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "eobhip_common.hpp"
#include "imr.hpp"
#include "resample.hpp"
#include "spline_nak.hpp"

using namespace eobhip_detail;
using imr::Cx;

namespace {

constexpr int kImrMaxModes = 8;
struct ImrModes {
    int nm;
    int l[kImrMaxModes];
    int m[kImrMaxModes];
};
constexpr int kImrMaxM = 5;     // the ringdown modes' largest m
constexpr int kImrAfter = 31;   // window rows kept past the evaluation interval
constexpr int kImrNqcBefore = 7; // rows before the NQC time (the reference's N = 7)
constexpr int kImrSeries = 7;   // q1 A, q2 A, q3 A, A, p1, p2, phase
constexpr double kTwoPi = 6.283185307179586;
constexpr double kPiD = 3.141592653589793;

// per (binary, mode) ringdown record
enum RdField { kRdAmp, kRdDamp, kRdPhi, kRdOmega, kRdC1c, kRdC2c, kRdC1f, kRdC2f, kRdD1c, kRdD1f, kRdD2f, kRdWr, kRdWi, kRdEta, kRdPad0, kRdPad1,
               kRdCount };
// per binary doubles and ints
enum BinField { kBinTPeak, kBinTMatch, kBinDt, kBinMf, kBinAf, kBinDT22, kBinCount };
enum BinInt { kBinNpts, kBinIdx, kBinNadd, kBinICount };

// t_k = k dT + t0 with the two roundings numpy makes (arange * delta_T + t_0)
__device__ __forceinline__ double grid_t(long long k, double dT, double t0) { return __dadd_rn(__dmul_rn((double)k, dT), t0); }

// argmin_k |t_k - T| over k < npts, first index on ties
__device__ int nearest_index(double T, double dT, double t0, int npts) {
    double kf = rint((T - t0) / dT);
    long long k = (kf == kf) ? (long long)fmax(fmin(kf, (double)(npts - 1)), 0.0) : 0;
    long long best = k;
    double bd = fabs(grid_t(k, dT, t0) - T);
    for (int d = -1; d <= 1; d += 2) {
        const long long kk = k + d;
        if (kk < 0 || kk >= npts) continue;
        const double dd = fabs(grid_t(kk, dT, t0) - T);
        if (dd < bd || (dd == bd && kk < best)) { best = kk; bd = dd; }
    }
    return (int)best;
}

// searchsorted(t_ws..t_{we-1}, T, 'right') - 1 as a grid index, clamped to [ws, we - 1]
__device__ int interval_index(double T, double dT, double t0, int ws, int we) {
    double kf = floor((T - t0) / dT);
    long long k = (kf == kf) ? (long long)fmax(fmin(kf, (double)(we - 1)), (double)ws) : ws;
    while (k > ws && grid_t(k, dT, t0) > T) --k;
    while (k + 1 < we && grid_t(k + 1, dT, t0) <= T) ++k;
    return (int)k;
}

// searchsorted(knots, t, 'right') - 1 over the binary's knots (row stride 5), >= 0
__device__ __forceinline__ int knot_index(const double* __restrict__ T, int len, double t) {
    int lo = 0, hi = len;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (T[5 * mid] <= t) lo = mid + 1;
        else hi = mid;
    }
    return lo > 0 ? lo - 1 : 0;
}

// A spline piece at offset x; the last knot's coefficients are zero (the
// reference fills knots 0 .. len - 2 only), so there the value is y and the
// derivative 0.
struct Piece {
    double x, x2, x3;
    bool last;
    __device__ static Piece at(double x, bool last) {
        const double x2 = x * x;
        return Piece{x, x2, x2 * x, last};
    }
    template <class Ptr>
    __device__ double v(Ptr c) const { return last ? c[0] : c[0] + c[1] * x + c[2] * x2 + c[3] * x3; }
    template <class Ptr>
    __device__ double d(Ptr c) const { return last ? 0.0 : c[1] + 2.0 * c[2] * x + 3.0 * c[3] * x2; }
};

// numpy.mod for a positive divisor
__device__ __forceinline__ double pymod(double x, double y) {
    double r = fmod(x, y);
    if (r != 0.0 && (r < 0.0) != (y < 0.0)) r += y;
    return r;
}

// numpy.unwrap over the wavefront's lanes 0 .. W - 1 (lane i holds sample i)
__device__ double unwrap_lanes(double ang, int lane, int W) {
    const double prev = __shfl_up(ang, 1, 64);
    double corr = 0.0;
    if (lane > 0 && lane < W) {
        const double dd = ang - prev;
        double ddmod = pymod(dd + kPiD, kTwoPi) - kPiD;
        if (ddmod == -kPiD && dd > 0.0) ddmod = kPiD;
        corr = (fabs(dd) < kPiD) ? 0.0 : ddmod - dd;
    }
    // inclusive prefix sum over the lanes
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(corr, off, 64);
        if (lane >= off) corr += o;
    }
    return ang + corr;
}

// Lane s < nser: the not-a-knot spline of series s over the W window samples
// (sh_t, sh_y[s]) evaluated at T in interval kI: value and first two
// derivatives (the reference's Thomas solve, src/interpolate.cu:11-267).
struct WinLds {
    double t[64];
    double y[kImrSeries][64];
    double ud[kImrSeries][64], dg[kImrSeries][64], b[kImrSeries][64];
    double val[kImrSeries][3];
};
__device__ void window_spline_eval(WinLds& w, int s, int W, int kI, double T) {
    const double* t = w.t;
    const double* y = w.y[s];
    double pdg = 0.0, pud = 0.0, pb = 0.0;
    for (int i = 0; i < W; ++i) {
        int i0, i1, i2;
        if (i == W - 1) { i0 = W - 3; i1 = W - 2; i2 = W - 1; }
        else if (i == 0) { i0 = 0; i1 = 1; i2 = 2; }
        else { i0 = i - 1; i1 = i; i2 = i + 1; }
        Row r = nak_row(i, W, t[i0], t[i1], t[i2], y[i0], y[i1], y[i2]);
        if (i > 0) {
            const double f = r.ld / pdg;
            r.dg = r.dg - f * pud;
            r.b = r.b - f * pb;
        }
        w.ud[s][i] = r.ud;
        w.dg[s][i] = r.dg;
        w.b[s][i] = r.b;
        pdg = r.dg; pud = r.ud; pb = r.b;
    }
    double sn = w.b[s][W - 1] / w.dg[s][W - 1];
    double s_hi = sn, s_lo = sn;
    for (int i = W - 2; i >= kI; --i) {
        s_hi = sn;
        sn = (w.b[s][i] - w.ud[s][i] * sn) / w.dg[s][i];
        s_lo = sn;
    }
    double c1 = 0.0, c2 = 0.0, c3 = 0.0;
    if (kI < W - 1) {
        const double dt = t[kI + 1] - t[kI];
        const double slope = (y[kI + 1] - y[kI]) / dt;
        const double tt = (s_lo + s_hi - 2.0 * slope) / dt;
        c1 = s_lo;
        c2 = (slope - s_lo) / dt - tt;
        c3 = tt / dt;
    }
    const double x = T - t[kI];
    w.val[s][0] = y[kI] + c1 * x + c2 * x * x + c3 * x * x * x;
    w.val[s][1] = c1 + 2.0 * c2 * x + 3.0 * c3 * x * x;
    w.val[s][2] = 2.0 * c2 + 6.0 * c3 * x;
}

// dense solves with partial pivoting (numpy.linalg.solve's LU), n <= 3
template <int N>
__device__ void solve_pivot(double A[N][N], double b[N], double x[N]) {
    for (int c = 0; c < N; ++c) {
        int p = c;
        for (int r = c + 1; r < N; ++r)
            if (fabs(A[r][c]) > fabs(A[p][c])) p = r;
        if (p != c) {
            for (int k = 0; k < N; ++k) { const double t = A[c][k]; A[c][k] = A[p][k]; A[p][k] = t; }
            const double t = b[c]; b[c] = b[p]; b[p] = t;
        }
        for (int r = c + 1; r < N; ++r) {
            const double f = A[r][c] / A[c][c];
            for (int k = c + 1; k < N; ++k) A[r][k] -= f * A[c][k];
            b[r] -= f * b[c];
        }
    }
    for (int r = N - 1; r >= 0; --r) {
        double s = b[r];
        for (int k = r + 1; k < N; ++k) s -= A[r][k] * x[k];
        x[r] = s / A[r][r];
    }
}

struct BinInputs {
    const double *m1, *m2, *chi1, *chi2;
};

// ------------------------------------------------------------- QNM table
// The five ringdown modes' roots (omega and the separation constant, Leaver
// units) on the spins -0.99 .. 0.99 in steps of 0.01, filled once per device;
// a binary's QNM is then a few secant steps from the interpolated entry
// instead of a walk from a = 0.  The mode index is imr::rd_mode_index.
constexpr int kQnmGrid = 199;
constexpr double kQnmA0 = -0.99, kQnmDa = 0.01;
__device__ double g_qnm_tab[5][kQnmGrid][4];

__device__ __forceinline__ void rd_mode_lm(int k, int& l, int& m) {
    l = (k <= 1) ? 2 : k + 1;
    m = (k == 1) ? 1 : l;
}

__global__ void k_qnm_table() {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 5 * kQnmGrid) return;
    const int k = t / kQnmGrid, i = t % kQnmGrid;
    int l, m;
    rd_mode_lm(k, l, m);
    const imr::QnmRoot r = imr::kerr_qnm_path(l, m, kQnmA0 + kQnmDa * i);
    double* o = g_qnm_tab[k][i];
    o[0] = r.w.re;
    o[1] = r.w.im;
    o[2] = r.A.re;
    o[3] = r.A.im;
}

// The fractions by 16 lanes (the same value, bit for bit, on all of them).  t_n =
// beta_n - alpha_n gamma_{n+1} / t_{n+1} is a Moebius map, so a lane multiplies the
// 2 x 2 matrices of its run of terms (no divisions) and four exchanges multiply
// the runs.  The radial maps are close to t -> -n^2 (2 + n^2 / t), whose products
// cancel: they act on t + n^2 instead, where what is left of alpha_n gamma_{n+1} is
// (n + 1)(c012 n^2 + e1 n + e0).  One secant step was 300 + 5 x 60 complex divisions
// in turn; 4096 roots 788 us, 119 now (91 without the steps below).
//
// The products' rounding stays in the root, where the division per term damps it on
// the way down: equal up to |a| = 0.8, but 1.5 to 2.5 times the serial error from
// there to 0.99.  There the root is corrected by the fraction with its lowest
// kLowTerms terms divided in turn (30 or more of them leave the serial rounding), and
// the mean of two such steps taken, of four from 0.97 on: the serial secant ends when
// two iterates agree by more than one evaluation's rounding, and so do these.  Rms of
// 1000 roots a mode against extended precision, serial, products alone and now, in
// 1e-16: (2,2) 4.4, 4.9, 3.5 from 0.8 on and 13, 32, 15 from 0.97 on; (5,5) 4.7, 6.7,
// 3.7 and 19, 40, 17.
constexpr int kQnmLanes = 16;
struct Moebius {
    Cx a, b, c, d;
};
__device__ __forceinline__ Cx mul_add(Cx x, Cx y, Cx z, Cx w) {
    return imr::cx(x.re * y.re - x.im * y.im + z.re * w.re - z.im * w.im, x.re * y.im + x.im * y.re + z.re * w.im + z.im * w.re);
}
// by a power of two to the size of 1
__device__ __forceinline__ void moebius_scale(Moebius& m) {
    const double s = fmax(fmax(fmax(fabs(m.a.re), fabs(m.a.im)), fmax(fabs(m.b.re), fabs(m.b.im))),
                          fmax(fmax(fabs(m.c.re), fabs(m.c.im)), fmax(fabs(m.d.re), fabs(m.d.im))));
    const double f = s > 0.0 && s < 1e300 ? ldexp(1.0, -ilogb(s)) : 1.0;
    m.a = f * m.a;
    m.b = f * m.b;
    m.c = f * m.c;
    m.d = f * m.d;
}
__device__ __forceinline__ Cx shfl_xor_cx(Cx v, int off) { return imr::cx(__shfl_xor(v.re, off, 64), __shfl_xor(v.im, off, 64)); }
// the lanes' product, applied to u
__device__ __forceinline__ Cx moebius_apply(Moebius m, Cx u) {
    moebius_scale(m);
#pragma unroll
    for (int off = 1; off < kQnmLanes; off <<= 1) {
        const Moebius o{shfl_xor_cx(m.a, off), shfl_xor_cx(m.b, off), shfl_xor_cx(m.c, off), shfl_xor_cx(m.d, off)};
        const bool up = threadIdx.x & off;
        const Moebius l = up ? o : m, h = up ? m : o;
        m = Moebius{mul_add(l.a, h.a, l.b, h.c), mul_add(l.a, h.b, l.b, h.d), mul_add(l.c, h.a, l.d, h.c), mul_add(l.c, h.b, l.d, h.d)};
        moebius_scale(m);
    }
    return (m.a * u + m.b) / (m.c * u + m.d);
}
struct LeaverLanes {
    __device__ static Cx fraction(const imr::LeaverAng& f) {
        constexpr int D = imr::kLeaverAngDepth, per = (D + kQnmLanes - 1) / kQnmLanes;
        const int lo = (int)(threadIdx.x % kQnmLanes) * per, hi = lo + per < D ? lo + per : D;
        Moebius m{imr::cx(1.0), imr::cx(0.0), imr::cx(0.0), imr::cx(1.0)};
#pragma unroll 1
        for (int n = hi - 1; n >= lo; --n) {
            const Cx be = imr::leaver_beta(f, n), g = -imr::leaver_alpha_gamma(f, n);
            m = Moebius{mul_add(be, m.a, g, m.c), mul_add(be, m.b, g, m.d), m.a, m.b};
        }
        return moebius_apply(m, imr::leaver_beta(f, D));
    }
    __device__ static Cx fraction(const imr::LeaverRad& f) { return radial_from<0>(f); }
    // t_K + K^2
    template <int K>
    __device__ static Cx radial_from(const imr::LeaverRad& f) {
        constexpr int D = imr::kLeaverRadDepth, per = (D - K + kQnmLanes - 1) / kQnmLanes;
        const int lo = K + (int)(threadIdx.x % kQnmLanes) * per, hi = lo + per < D ? lo + per : D;
        const Cx p = f.c1 + 2.0, e1 = p + f.c3 + f.c4 + f.c0 * (f.c2 - 1.0), e0 = f.c3 + f.c0 * f.c4;
        Moebius m{imr::cx(1.0), imr::cx(0.0), imr::cx(0.0), imr::cx(1.0)};
#pragma unroll 1
        for (int n = hi - 1; n >= lo; --n) {
            const double d = n, e = d + 1.0;
            const Cx h = p * d + f.c3 - d * d, g = (-e) * ((f.c012 * d + e1) * d + e0);
            m = Moebius{mul_add(h, m.a, g, m.c), mul_add(h, m.b, g, m.d), m.a - (e * e) * m.c, m.b - (e * e) * m.d};
        }
        const double d = D;
        return moebius_apply(m, p * d + f.c3 - d * d);
    }
};

constexpr int kLowTerms = 40;

// M omega_lm0 at spin |af| <= 0.99 of a ringdown mode, from the table's guess; Cf
// LeaverLanes: by the kQnmLanes lanes of a group
template <class Cf>
__device__ Cx kerr_qnm_table(int k, int m, double af) {
    const double x = (af - kQnmA0) / kQnmDa;
    int i = (int)floor(x);
    i = i < 0 ? 0 : (i > kQnmGrid - 2 ? kQnmGrid - 2 : i);
    const double f = x - i;
    const double* p0 = g_qnm_tab[k][i];
    const double* p1 = g_qnm_tab[k][i + 1];
    const Cx w = imr::cx((1.0 - f) * p0[0] + f * p1[0], (1.0 - f) * p0[1] + f * p1[1]);
    const Cx A = imr::cx((1.0 - f) * p0[2] + f * p1[2], (1.0 - f) * p0[3] + f * p1[3]);
    imr::QnmRoot r = imr::leaver_refine<Cf>(m, 0.5 * af, w, A, 1e-6);
    if constexpr (std::is_same_v<Cf, LeaverLanes>) {
        if (fabs(af) >= 0.8) {
            const double a = 0.5 * af;
            const int steps = fabs(af) < 0.97 ? 2 : 4;
            Cx sum = imr::cx(0.0);
#pragma unroll 1
            for (int k = 0; k < steps; ++k) {
                if (k) r.A = imr::leaver_angular_solve<LeaverLanes>(r.A, a * r.w, -2, m);
                const imr::LeaverRad f = imr::leaver_radial(r.w, a, -2, m, r.A);
                const Cx t = LeaverLanes::radial_from<kLowTerms>(f) - (double)(kLowTerms * kLowTerms);
                r.w = r.w - r.slope * imr::leaver_radial_down(f, t, kLowTerms);
                sum = sum + r.w;
            }
            r.w = (1.0 / steps) * sum;
        }
    }
    return imr::cx(0.5 * r.w.re, 0.5 * r.w.im);
}

// How a launch of blocks of 64 threads shares n roots: in its first `groups` blocks a
// group of kQnmLanes lanes per root that the table serves, in the others a lane per
// root for what is left: roots without a table (the spin path from a = 0, where a
// group's lanes would all walk the same path) and, with no groups, all.  Up to
// kQnmGrouped roots the groups are faster, since a root's chain is the time: (2,2),
// 4096 roots 118 us by groups and 785 by lanes, 65536 926 and 771, 262144 3444 and 2036.
// Without a table, 65536 roots 16.5 ms a lane each and 101 by groups.
constexpr long long kQnmGrouped = 49152;
struct QnmSplit {
    unsigned groups;
    static QnmSplit of(long long n, bool table) { return QnmSplit{table && n <= kQnmGrouped ? blocks_for(n, 64 / kQnmLanes) : 0u}; }
    unsigned blocks(long long n) const { return groups + blocks_for(n, 64); }
    __device__ __forceinline__ bool grouped() const { return blockIdx.x < groups; }
    __device__ __forceinline__ long long root() const {
        return grouped() ? ((long long)blockIdx.x * 64 + threadIdx.x) / kQnmLanes : (long long)(blockIdx.x - groups) * 64 + threadIdx.x;
    }
    // M omega_lm0 at spin af; true on the one lane that has it
    __device__ __forceinline__ bool omega(int l, int m, double af, Cx& w) const {
        const int k = imr::rd_mode_index(l, m);
        const bool table = k >= 0 && fabs(af) <= 0.99;
        if (grouped()) {
            if (table) w = kerr_qnm_table<LeaverLanes>(k, m, af);
            return table && threadIdx.x % kQnmLanes == 0;
        }
        if (table && groups) return false;
        w = table ? kerr_qnm_table<imr::LeaverSerial>(k, m, af) : imr::kerr_qnm(l, m, af);
        return true;
    }
};

// fill the table on the current device once (stream-ordered, then waited for,
// so that launches on any stream see it)
std::mutex g_qnm_mu;
bool g_qnm_ready[64];
int ensure_qnm_table(void* stream) {
    int dev = 0;
    int rc = hip_status(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    std::lock_guard<std::mutex> lk(g_qnm_mu);
    if (dev >= 0 && dev < 64 && g_qnm_ready[dev]) return EOBHIP_OK;
    hipLaunchKernelGGL(k_qnm_table, dim3(blocks_for(5 * kQnmGrid, 64)), dim3(64), 0, as_stream(stream));
    rc = check_launch("qnm_table");
    if (rc) return rc;
    rc = hip_status(hipStreamSynchronize(as_stream(stream)), "qnm_table sync");
    if (rc) return rc;
    if (dev >= 0 && dev < 64) g_qnm_ready[dev] = true;
    return EOBHIP_OK;
}

// ------------------------------------------------------------ QNMs per binary
// Root (b, j): j < nm the QNM of mode j, j == nm the (2,2) QNM that sets the
// ringdown length (the reference's 30 damping times, :2463-2465 and :2514).
// wl [n][nm] complex in lalsimulation's convention (omega_r + i / tau) in
// units of the total mass; binf/bini as the enums.
__global__ void k_imr_qnm(BinInputs in, const double* __restrict__ dense, const double* __restrict__ dT_M, int n, int max_step,
                          ImrModes mm, QnmSplit split, double* __restrict__ wl, double* __restrict__ binf, int* __restrict__ bini) {
    const long long gid = split.root();
    const int per = mm.nm + 1;
    if (gid >= (long long)n * per) return;
    const int b = (int)(gid / per), j = (int)(gid % per);
    const double m1 = in.m1[b], m2 = in.m2[b], c1 = in.chi1[b], c2 = in.chi2[b];
    const double M = m1 + m2;
    const double mf = imr::final_mass_seobnrv4(m1 / M, m2 / M, c1, c2);
    const double af = imr::final_spin_hbr2016(m1 / M, m2 / M, c1, c2);
    const int l = (j < mm.nm) ? mm.l[j] : 2, m = (j < mm.nm) ? mm.m[j] : 2;
    Cx w;
    if (!split.omega(l, m, af, w)) return;
    const double wr = w.re / mf, wi = -w.im / mf;   // conj(omega) / M_f
    if (j < mm.nm) {
        wl[2 * ((size_t)b * mm.nm + j)] = wr;
        wl[2 * ((size_t)b * mm.nm + j) + 1] = wi;
        return;
    }
    binf[(size_t)b * kBinCount + kBinMf] = mf;
    binf[(size_t)b * kBinCount + kBinAf] = af;
    const double t0 = dense[(size_t)b * max_step * 5];
    const double dT = dT_M[b];
    const double dt = grid_t(1, dT, t0) - grid_t(0, dT, t0);
    const double ringdown_time = trunc(30.0 * (1.0 / wi));
    const double nadd = floor(ringdown_time / dt) + 1.0;
    bini[(size_t)b * kBinICount + kBinNadd] = (dt > 0.0 && nadd >= 1.0 && nadd < 1073741824.0) ? (int)nadd : 0;
}

// ------------------------------------------------ NQC and ringdown parameters
// One wavefront per (binary, mode): block b * nm + q.
__global__ __launch_bounds__(64) void k_imr_params(BinInputs in, const double* __restrict__ dense, const int* __restrict__ num_steps,
                                                   const double* __restrict__ coef, const double* __restrict__ rp,
                                                   const double* __restrict__ dT_M, int max_step, ImrModes mm,
                                                   const double* __restrict__ wl, double* __restrict__ nqc, double* __restrict__ rd,
                                                   double* __restrict__ binf, int* __restrict__ bini) {
    __shared__ WinLds w;
    const int b = blockIdx.x / mm.nm, q = blockIdx.x % mm.nm;
    const int lane = threadIdx.x;
    const int nm = mm.nm, cs = 4 * (2 * nm + 1);
    const int l = mm.l[q], m = mm.m[q];
    const int len = num_steps[b];
    double* out_nqc = nqc + ((size_t)b * nm + q) * 5;
    double* out_rd = rd + ((size_t)b * nm + q) * kRdCount;
    const double* T = dense + (size_t)b * max_step * 5;
    const double* C = coef + (size_t)b * max_step * cs;
    const double* RP = rp + (size_t)b * max_step * 8;
    const double t0 = T[0];
    const double dT = dT_M[b];
    // grid samples up to the last knot (a spacing that is not positive, or a
    // grid beyond 2^30 samples, marks the binary as failed)
    const double span = (len >= 1 && dT > 0.0) ? (T[5 * (len - 1)] - t0) / dT : -1.0;
    const int npts = (span >= 0.0 && span < 1073741824.0) ? (int)span + 1 : 0;
    if (len < 4 || npts < 2 * kImrAfter + 16) {
        if (lane < 5) out_nqc[lane] = NAN;
        if (lane < kRdCount) out_rd[lane] = NAN;
        if (q == 0 && lane == 0) {
            bini[(size_t)b * kBinICount + kBinNpts] = npts;
            bini[(size_t)b * kBinICount + kBinIdx] = -1;
        }
        return;
    }
    // time of the orbital-frequency peak over the knots (phi's slope at the
    // knots, 0 at the last one; first maximum)
    double best = -INFINITY;
    int bi = 0;
    for (int i = lane; i < len; i += 64) {
        const double v = (i < len - 1) ? C[(size_t)cs * i + 4 * (2 * nm) + 1] : 0.0;
        if (v > best) { best = v; bi = i; }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double ob = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    const double t_peak = T[5 * bi];
    const imr::FitIn fin{in.m1[b], in.m2[b], in.chi1[b], in.chi2[b]};
    const double dT22 = imr::nr_peak_delta_t(fin);
    const bool is55 = (l == 5 && m == 5);

    // sample window [ws, we) of the grid: the mode h, |h|, unwrapped phase, r, pr, omega (one sample per lane)
    auto sample = [&](int k, double& hr, double& hi, double& r, double& pr, double& om) {
        const double tk = grid_t(k, dT, t0);
        const int ind = knot_index(T, len, tk);
        Piece p;
        p.x = tk - T[5 * ind];
        p.x2 = p.x * p.x;
        p.x3 = p.x2 * p.x;
        p.last = (ind == len - 1);
        const double* row = C + (size_t)cs * ind;
        const double phi = p.v(row + 4 * (2 * nm));
        om = p.d(row + 4 * (2 * nm));
        const double re = p.v(row + 4 * q), im = p.v(row + 4 * (nm + q));
        r = p.v(RP + (size_t)8 * ind);
        pr = p.v(RP + (size_t)8 * ind + 4);
        double s, c;
        sincos((double)m * phi, &s, &c);
        hr = re * c + im * s;
        hi = im * c - re * s;
    };

    // ---- NQC (EOBCalculateNQCCoefficientsV4_freeattach)
    const double Tn = t_peak - dT22 - (is55 ? 10.0 : 0.0);
    const int idx = nearest_index(Tn, dT, t0, npts);
    const int ws = idx - kImrNqcBefore > 0 ? idx - kImrNqcBefore : 0;
    const int kI = interval_index(Tn, dT, t0, ws, npts);
    const int we = (kI + kImrAfter + 1 < npts) ? kI + kImrAfter + 1 : npts;
    const int W = we - ws;
    {
        double hr = 0.0, hi = 0.0, r = 1.0, pr = 0.0, om = 1.0;
        if (lane < W) sample(ws + lane, hr, hi, r, pr, om);
        const double amp = hypot(hr, hi);
        const double ph = unwrap_lanes(atan2(hi, hr), lane, W);
        if (lane < W) {
            const double rO = r * om;
            const double q1 = pr * pr / (rO * rO);
            const double q2 = q1 / r;
            const double q3 = q2 / sqrt(r);
            const double p1 = pr / rO;
            w.t[lane] = grid_t(ws + lane, dT, t0);
            w.y[0][lane] = q1 * amp;
            w.y[1][lane] = q2 * amp;
            w.y[2][lane] = q3 * amp;
            w.y[3][lane] = amp;
            w.y[4][lane] = p1;
            w.y[5][lane] = p1 * pr * pr;
            w.y[6][lane] = ph;
        }
    }
    __syncthreads();
    if (lane < kImrSeries) window_spline_eval(w, lane, W, kI - ws, Tn);
    __syncthreads();
    double nq[5];
    {
        double Q[3][3], rhs[3], a[3];
        for (int i = 0; i < 3; ++i)
            for (int k = 0; k < 3; ++k) Q[i][k] = w.val[k][i];
        rhs[0] = fabs(imr::nr_peak_amp(l, m, fin)) - w.val[3][0];
        rhs[1] = imr::nr_peak_adot(l, m, fin) - w.val[3][1];
        rhs[2] = imr::nr_peak_addot(l, m, fin) - w.val[3][2];
        solve_pivot<3>(Q, rhs, a);
        double P[2][2], r2[2], bb[2];
        for (int i = 1; i <= 2; ++i) {
            P[i - 1][0] = -w.val[4][i];
            P[i - 1][1] = -w.val[5][i];
        }
        const double wt = w.val[6][1], wdt = w.val[6][2];
        const double omega = fabs(wt);
        const double omegaDot = (wt * wdt > 0.0) ? fabs(wdt) : -fabs(wdt);
        const double eta = fin.m1 * fin.m2 / ((fin.m1 + fin.m2) * (fin.m1 + fin.m2));
        const double chi = imr::fit_chi(fin);
        r2[0] = imr::nr_peak_omega(l, m, eta, chi) - omega;
        r2[1] = imr::nr_peak_omegadot(l, m, eta, chi) - omegaDot;
        solve_pivot<2>(P, r2, bb);
        nq[0] = a[0]; nq[1] = a[1]; nq[2] = a[2]; nq[3] = bb[0]; nq[4] = bb[1];
    }
    if (lane < 5) out_nqc[lane] = nq[lane];
    __syncthreads();   // the window is rewritten below

    // ---- ringdown attachment (compute_full_waveform :2438-2519, compute_MR_mode_free)
    const double t_attach = t_peak - dT22;
    const int idr = nearest_index(t_attach, dT, t0, npts);
    const double dt = grid_t(1, dT, t0) - grid_t(0, dT, t0);
    const long long Nw = (long long)(20.0 / dt) + 1;
    const double t_match = grid_t(idr, dT, t0);
    const double tm = t_match - (is55 ? 10.0 : 0.0);
    const int ws2 = (idr - Nw > 0) ? (int)(idr - Nw) : 0;
    const int kR = interval_index(tm, dT, t0, ws2, npts);
    const int wlo = (kR - kImrAfter > ws2) ? kR - kImrAfter : ws2;
    const int whi = (kR + kImrAfter + 1 < npts) ? kR + kImrAfter + 1 : npts;
    const int W2 = whi - wlo;
    {
        double hr = 0.0, hi = 0.0, r = 1.0, pr = 0.0, om = 1.0;
        if (lane < W2) sample(wlo + lane, hr, hi, r, pr, om);
        // the NQC factor (EOBNonQCCorrection with a3S = a4 = a5 = b3 = b4 = 0)
        const double sr = sqrt(r), rO = r * om;
        const double mag = 1.0 + (pr * pr / (rO * rO)) * (nq[0] + nq[1] / r + nq[2] / (r * sr));
        const double nph = nq[3] * pr / rO + pr * pr * pr / rO * nq[4];
        double sn, cn;
        sincos(nph, &sn, &cn);
        const double fr = mag * cn, fi = mag * sn;
        const double cr = hr * fr - hi * fi, ci = hr * fi + hi * fr;
        const double amp = hypot(cr, ci);
        const double ph = unwrap_lanes(atan2(ci, cr), lane, W2);
        if (lane < W2) {
            w.t[lane] = grid_t(wlo + lane, dT, t0);
            w.y[0][lane] = amp;
            w.y[1][lane] = ph;
        }
    }
    __syncthreads();
    if (lane < 2) window_spline_eval(w, lane, W2, kR - wlo, tm);
    __syncthreads();
    if (lane == 0) {
        const double A0 = w.val[0][0], dA0 = w.val[0][1], phm = w.val[1][0], wm = w.val[1][1];
        const double wr = wl[2 * ((size_t)b * nm + q)], wi = wl[2 * ((size_t)b * nm + q) + 1];
        const double sR = -wi, sI = -wr;
        const double eta = fin.m1 * fin.m2 / ((fin.m1 + fin.m2) * (fin.m1 + fin.m2));
        const double chi = imr::fit_chi(fin);
        const int ri = imr::rd_mode_index(l, m);
        double c1f = NAN, c2f = NAN, d1f = NAN, d2f = NAN;
        if (ri >= 0) {
            c1f = imr::rd_poly(imr::rd_table_a1(ri), eta, chi);
            c2f = imr::rd_poly(imr::rd_table_a2(ri), eta, chi);
            d1f = imr::rd_poly(imr::rd_table_p1(ri), eta, chi);
            d2f = imr::rd_poly(imr::rd_table_p2(ri), eta, chi);
        }
        if (ri == 0 && sR > 2.0 * c1f * tanh(c2f)) c1f = sR / (2.0 * tanh(c2f));
        const double ch = cosh(c2f);
        const double c1c = 1.0 / (c1f * eta) * (dA0 - sR * A0) * ch * ch;
        const double c2c = A0 / eta - 1.0 / (c1f * eta) * (dA0 - sR * A0) * ch * sinh(c2f);
        const double d1c = (wm - sI) * (1.0 + d2f) / (d1f * d2f);
        double* o = out_rd;
        o[kRdAmp] = A0; o[kRdDamp] = dA0; o[kRdPhi] = phm; o[kRdOmega] = wm;
        o[kRdC1c] = c1c; o[kRdC2c] = c2c; o[kRdC1f] = c1f; o[kRdC2f] = c2f;
        o[kRdD1c] = d1c; o[kRdD1f] = d1f; o[kRdD2f] = d2f;
        o[kRdWr] = wr; o[kRdWi] = wi; o[kRdEta] = eta; o[kRdPad0] = 0.0; o[kRdPad1] = 0.0;
        if (q == 0) {
            double* bf = binf + (size_t)b * kBinCount;
            bf[kBinTPeak] = t_peak;
            bf[kBinTMatch] = t_match;
            bf[kBinDt] = dt;
            bf[kBinDT22] = dT22;
            bini[(size_t)b * kBinICount + kBinNpts] = npts;
            bini[(size_t)b * kBinICount + kBinIdx] = idr;
        }
    }
}

// sin and cos of x: Taylor series through x^9 / x^10 when every active lane of
// the wavefront has |x| < 1/16 (first omitted terms below 2.3e-20 relative),
// sincos_of otherwise.  The NQC phase of the inspiral samples is small except near the
// attachment.
template <Phases P>
__device__ __forceinline__ bool sincos_nqc(double x, double* s, double* c) {
    if (__all(fabs(x) < 0.0625)) {
        const double x2 = x * x;
        *s = x * (1.0 + x2 * (-1.0 / 6 + x2 * (1.0 / 120 + x2 * (-1.0 / 5040 + x2 * (1.0 / 362880)))));
        *c = 1.0 + x2 * (-0.5 + x2 * (1.0 / 24 + x2 * (-1.0 / 720 + x2 * (1.0 / 40320 + x2 * (-1.0 / 3628800)))));
        return true;
    }
    return sincos_of<P>(x, *s, *c);
}

// ------------------------------------------------------- the IMR template
// h_j = amp (sum over modes of h_lm NQC_lm (t_j) for j <= idx, of the ringdown
// for idx < j < idx + nadd, 0 after), t_j = t_0 + j dT; hplus = Re, hcross = Im.
constexpr int kImrBlock = 256;
constexpr int kRingBlocks = 4;   // blocks on a binary's ringdown

// One inspiral sample's sum over the modes: row holds the interval's spline
// coefficients (Re of each mode, Im of each mode, phi), rpr those of r and pr; nq
// the binary's NQC coefficients (5 per mode).  sum_m h_m e^{-i m phi} by Horner's
// rule in e^{-i phi} over the modes by falling m (mo): each mode then costs the
// products between its m and the next one's, not m - 1 of its own.
template <Phases kPath, class Ptr>
__device__ __forceinline__ bool imr_inspiral_sample(Ptr row, Ptr rpr, const Piece& p, int nm, const ModeOrder& mo, const double* nq,
                                                    double& re_out, double& im_out) {
    const double om = p.d(row + 4 * (2 * nm)), r = p.v(rpr), pr = p.v(rpr + 4);
    // each rounded once: the NQC coefficients come from nearly singular solves and
    // cancel in the sums below by up to eight digits
    const double rO = r * om, ir = 1.0 / r, irs = 1.0 / (r * sqrt(r));
    const double p1 = pr / rO, p3 = pr * pr * pr / rO, P = p1 * p1;
    double sp, cph, hr = 0.0, hi = 0.0;
    bool good = sincos_of<kPath>(p.v(row + 4 * (2 * nm)), sp, cph);
    const auto turn = [&](int k) {
        for (; k > 0; --k) {
            const double t = hr * cph + hi * sp;
            hi = hi * cph - hr * sp;
            hr = t;
        }
    };
#pragma unroll 1
    for (int k = 0; k < nm; ++k) {
        const int q = mo.q(k);
        const Ptr rq = row + 4 * q, iq = row + 4 * (nm + q);
        const double* c = nq + 5 * q;
        double sn, cn;
        good &= sincos_nqc<kPath>(c[3] * p1 + p3 * c[4], &sn, &cn);
        turn(mo.down(k));
        const double mag = 1.0 + P * (c[0] + c[1] * ir + c[2] * irs);
        const double re = p.v(rq), im = p.v(iq), fr = mag * cn, fi = mag * sn;
        hr += re * fr - im * fi;
        hi += re * fi + im * fr;
    }
    turn(mo.down(nm));
    re_out = hr;
    im_out = hi;
    return good;
}

// samples of a template: inspiral 0 .. idx, ringdown to idx + nadd; 0: none
__device__ __forceinline__ long long imr_samples(int idx, int nadd, int len) {
    return (idx < 0 || len < 4) ? 0 : (long long)idx + (nadd > 0 ? nadd : 1);
}

// The ringdown of a binary (rd: its modes' rows of kRdCount), the sum over the modes
// at sample j > idx
struct Ringdown {
    const double* rd;
    double t_match, dt;
    long long idx;
    __device__ __forceinline__ void sample(long long j, int nm, double& hr, double& hi) const {
        const double x = (t_match + (double)(j - idx) * dt) - t_match;
        hr = hi = 0.0;
        for (int q = 0; q < nm; ++q) {
            const double* o = rd + (size_t)q * kRdCount;
            const double Alm = o[kRdC1c] * tanh(o[kRdC1f] * x + o[kRdC2f]) + o[kRdC2c];
            const double philm = o[kRdPhi] - o[kRdD1c] * log((1.0 + o[kRdD2f] * exp(-o[kRdD1f] * x)) / (1.0 + o[kRdD2f]));
            const double mod = o[kRdEta] * Alm * exp(-o[kRdWi] * x);
            double s, c;
            sincos(philm - o[kRdWr] * x, &s, &c);
            hr += mod * c;
            hi += mod * s;
        }
    }
};

// grid (blocks, binaries), runs of samples per wavefront (resample.hpp).  512
// binaries x 2^20 samples at 16384 Hz, five modes, 32% of them inspiral: 6100 us
// with knot windows per block and ten complex products a sample, 3350 now.  The
// arithmetic alone is about 1750 (375 instructions a sample at the FP64 rate; with
// one shared reciprocal for its four divisions and the root 1540 and 3055, but an
// ulp or two off where the NQC sums cancel) and the writes 1360: a binary's blocks run together, so
// the two hardly overlap (taking the binaries in turn instead scatters the writes
// and costs a fifth more).  Three wavefronts a SIMD; four (spills) or two samples at once
// (two wavefronts) are no faster.
//
// A binary's last kRingBlocks blocks take its ringdown, which the others leave out.
// (Its few hundred samples in a launch of their own: 20 us for 17 where one binary
// of 2^18 samples and one mode is the batch, 34 for 28 with five modes, 280 for 260
// with 256 binaries of 2^16; by the lanes that would write zeros there: 23, 47 and 386.)
// One build for any number of modes: 23 table rows of five are staged, 16 of eight (with
// 8 rows 64 binaries x 2^14 of eight modes 44.9 us, 41.9 now; 21 rows are no faster).
constexpr int kImrRoom = 1280;   // a wavefront's doubles of LDS
template <int kRows>
__global__ __launch_bounds__(kImrBlock) void k_imr_resample(const double* __restrict__ dense, const int* __restrict__ num_steps,
                                                            const double* __restrict__ coef, const double* __restrict__ rp,
                                                            const double* __restrict__ amp, const double* __restrict__ dT_M, int max_step,
                                                            int N, int nm, ModeOrder mo, const double* __restrict__ nqc,
                                                            const double* __restrict__ rd, const double* __restrict__ binf,
                                                            const int* __restrict__ bini, double* __restrict__ hplus,
                                                            double* __restrict__ hcross, int* __restrict__ nsamp) {
    const int cs = 4 * (2 * nm + 1);
    const int b = blockIdx.y;
    const int len = num_steps[b];
    const int idx = bini[(size_t)b * kBinICount + kBinIdx];
    const int nadd = bini[(size_t)b * kBinICount + kBinNadd];
    const long long nvalid = imr_samples(idx, nadd, len);
    if (blockIdx.x == 0 && threadIdx.x == 0) nsamp[b] = (int)(nvalid < N ? nvalid : N);
    const long long jinsp = nvalid == 0 ? 0 : ((long long)idx + 1 < N ? (long long)idx + 1 : N);   // inspiral samples j < jinsp
    const double* T = dense + (size_t)b * max_step * 5;
    const double* C = coef + (size_t)b * max_step * cs;
    const double* RP = rp + (size_t)b * max_step * 8;
    const double t0 = T[0], dT = dT_M[b];
    const long long stop = nvalid < N ? nvalid : N;
    const SeriesOut<true> o{hplus + (size_t)b * N, hcross + (size_t)b * N, amp[b], jinsp, N, stop};   // nvalid >= idx + 1, or 0
    // Blocks go to the eight XCDs in turn: in a grid of 8 k a row, each binary's ringdown
    // would be on the same four, so that the rows take turns too (512 binaries x 2^13, one and
    // five modes: 95 and 154 us, 57 and 93 in turn; where the grid is another, 64 x 2^14 33 and
    // 37 in turn).
    const unsigned blocks = gridDim.x - kRingBlocks, block = gridDim.x % 8 ? blockIdx.x : (blockIdx.x + blockIdx.y) % gridDim.x;
    if (block >= blocks) {
        const double t_match = binf[(size_t)b * kBinCount + kBinTMatch], dt = binf[(size_t)b * kBinCount + kBinDt];
        const Ringdown ring{rd + (size_t)b * nm * kRdCount, t_match, dt, idx};
        for (long long j = idx + 1 + (long long)(block - blocks) * blockDim.x + threadIdx.x; j < stop; j += kRingBlocks * blockDim.x) {
            double hr, hi;
            ring.sample(j, nm, hr, hi);
            o.out[j] = o.a * hr;
            o.outc[j] = o.a * hi;
        }
        return;
    }
    // a wavefront's NQC factors and table rows: the modes', then those of rp
    extern __shared__ __attribute__((aligned(16))) double staged[];
    const int most = staged_rows(kImrRoom - 5 * kImrMaxModes, cs + 8);
    double *nq = staged + wave_index() * kImrRoom, *ms = nq + 5 * kImrMaxModes, *rs = ms + most * cs;
    if ((int)(threadIdx.x & 63) < 5 * nm) nq[threadIdx.x & 63] = nqc[(size_t)b * nm * 5 + (threadIdx.x & 63)];
    for_runs(N, kRows, block, blocks, [&](long long j0) {
        if (j0 < jinsp)
            resample_rows(
                kRows, most, true, T, len, j0, jinsp, [&](long long j) { return grid_t(j, dT, t0); },
                [&](int i, int n) {
                    stage_rows<5>(ms, C + (size_t)cs * i, n, cs);
                    stage_rows<1>(rs, RP + (size_t)8 * i, n, 8);
                    if (i + n == len) {   // the last knot's interval: its value, no slope
                        __builtin_amdgcn_wave_barrier();
                        flatten_row(ms + (n - 1) * cs, cs);
                        flatten_row(rs + (n - 1) * 8, 8);
                    }
                },
                [&](int k, double x, double& re, double& im) {
                    return imr_inspiral_sample<kBounded>(ms + k * cs, rs + 8 * k, Piece::at(x, false), nm, mo, nq, re, im);
                },
                [&](int i, double x, double& re, double& im) {
                    return imr_inspiral_sample<kBounded>(C + (size_t)cs * i, RP + (size_t)8 * i, Piece::at(x, i == len - 1), nm, mo, nq, re, im);
                },
                [&](int i, double x, double& re, double& im) {
                    return imr_inspiral_sample<kAny>(C + (size_t)cs * i, RP + (size_t)8 * i, Piece::at(x, i == len - 1), nm, mo, nq, re, im);
                },
                [&](long long j, const double (&re)[2], const double (&im)[2], bool full) { o.put(j, re, im, full); });
        o.zeros(j0, kRows);
    });
}

// ---------------------------------------------------------- drop-in fits
__global__ void k_imr_fit(int which, int l, int m, const double* __restrict__ x1, const double* __restrict__ x2,
                          const double* __restrict__ x3, const double* __restrict__ x4, int n, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double a = x1[i], b = x2 ? x2[i] : 0.0, c = x3 ? x3[i] : 0.0, d = x4 ? x4[i] : 0.0;
    double v = NAN;
    switch (which) {
        case EOBHIP_FIT_DT22: v = imr::nr_peak_delta_t({a, b, c, d}); break;
        // amplitude fits take (m1, m2, chiS, chiA) as the reference's functions do
        case EOBHIP_FIT_AMP: v = imr::nr_peak_amp(l, m, {a, b, c + d, c - d}); break;
        case EOBHIP_FIT_ADOT: v = imr::nr_peak_adot(l, m, {a, b, c + d, c - d}); break;
        case EOBHIP_FIT_ADDOT: v = imr::nr_peak_addot(l, m, {a, b, c + d, c - d}); break;
        case EOBHIP_FIT_OMEGA: v = imr::nr_peak_omega(l, m, a, b); break;
        case EOBHIP_FIT_OMEGADOT: v = imr::nr_peak_omegadot(l, m, a, b); break;
        case EOBHIP_FIT_C1F: { const int k = imr::rd_mode_index(l, m); if (k >= 0) v = imr::rd_poly(imr::rd_table_a1(k), a, b); } break;
        case EOBHIP_FIT_C2F: { const int k = imr::rd_mode_index(l, m); if (k >= 0) v = imr::rd_poly(imr::rd_table_a2(k), a, b); } break;
        case EOBHIP_FIT_D1F: { const int k = imr::rd_mode_index(l, m); if (k >= 0) v = imr::rd_poly(imr::rd_table_p1(k), a, b); } break;
        case EOBHIP_FIT_D2F: { const int k = imr::rd_mode_index(l, m); if (k >= 0) v = imr::rd_poly(imr::rd_table_p2(k), a, b); } break;
        case EOBHIP_FIT_FINAL_MASS: v = imr::final_mass_seobnrv4(a, b, c, d); break;
        case EOBHIP_FIT_FINAL_SPIN: v = imr::final_spin_hbr2016(a, b, c, d); break;
        case EOBHIP_FIT_ISCO_RADIUS: v = imr::kerr_isco_radius(a); break;
        default: break;
    }
    out[i] = v;
}

__global__ void k_kerr_qnm(int l, int m, const double* __restrict__ af, int n, QnmSplit split, double* __restrict__ out) {
    const long long i = split.root();
    if (i >= n) return;
    Cx w;
    if (!split.omega(l, m, af[i], w)) return;
    out[2 * i] = w.re;
    out[2 * i + 1] = w.im;
}

int make_modes(ImrModes& mm, int nm, const int* ls, const int* ms) {
    EOBHIP_REQUIRE(nm >= 1 && nm <= kImrMaxModes, "1 <= nm <= %d", kImrMaxModes);
    mm.nm = nm;
    for (int i = 0; i < nm; ++i) {
        EOBHIP_REQUIRE(imr::rd_mode_index(ls[i], ms[i]) >= 0, "mode (%d, %d) has no ringdown fit", ls[i], ms[i]);
        mm.l[i] = ls[i];
        mm.m[i] = ms[i];
    }
    return EOBHIP_OK;
}

}  // namespace

extern "C" {

int eobhip_imr_fit(int which, int l, int m, const double* x1, const double* x2, const double* x3, const double* x4, int n, double* out,
                   void* stream) {
    EOBHIP_REQUIRE(n >= 0 && which >= 0 && which < EOBHIP_FIT_COUNT, "bad arguments");
    if (n == 0) return EOBHIP_OK;
    hipLaunchKernelGGL(k_imr_fit, dim3(blocks_for(n, 128)), dim3(128), 0, as_stream(stream), which, l, m, x1, x2, x3, x4, n, out);
    return check_launch("imr_fit");
}

int eobhip_kerr_qnm(int l, int m, const double* af, int n, double* omega, void* stream) {
    EOBHIP_REQUIRE(n >= 0 && l >= 2 && l <= 5 && m >= -l && m <= l && l == (abs(m) > 2 ? abs(m) : 2),
                   "bad arguments (the fundamental mode of l = max(2, |m|), l <= 5)");
    if (n == 0) return EOBHIP_OK;
    const int rc = ensure_qnm_table(stream);
    if (rc) return rc;
    const QnmSplit split = QnmSplit::of(n, imr::rd_mode_index(l, m) >= 0);
    hipLaunchKernelGGL(k_kerr_qnm, dim3(split.blocks(n)), dim3(64), 0, as_stream(stream), l, m, af, n, split, omega);
    return check_launch("kerr_qnm");
}

int eobhip_imr_params(const double* m1, const double* m2, const double* chi1, const double* chi2, const double* dense,
                      const int* num_steps, const double* coef, const double* rp_coef, const double* dT_M, int n, int max_step, int nm,
                      const int* ls, const int* ms, double* qnm, double* nqc, double* rd, double* binf, int* bini, void* stream) {
    ImrModes mm;
    int rc = make_modes(mm, nm, ls, ms);
    if (rc) return rc;
    EOBHIP_REQUIRE(n >= 0 && max_step >= 4, "bad sizes");
    if (n == 0) return EOBHIP_OK;
    rc = ensure_qnm_table(stream);
    if (rc) return rc;
    const BinInputs in{m1, m2, chi1, chi2};
    const long long nq = (long long)n * (nm + 1);
    const QnmSplit split = QnmSplit::of(nq, true);
    hipLaunchKernelGGL(k_imr_qnm, dim3(split.blocks(nq)), dim3(64), 0, as_stream(stream), in, dense, dT_M, n, max_step, mm, split, qnm, binf, bini);
    rc = check_launch("imr_qnm");
    if (rc) return rc;
    EOBHIP_REQUIRE((long long)n * nm < (1LL << 31), "too many (binary, mode) pairs");
    hipLaunchKernelGGL(k_imr_params, dim3(n * nm), dim3(64), 0, as_stream(stream), in, dense, num_steps, coef, rp_coef, dT_M, max_step, mm,
                       qnm, nqc, rd, binf, bini);
    return check_launch("imr_params");
}

int eobhip_imr_resample(const double* dense, const int* num_steps, const double* coef, const double* rp_coef, const double* amp,
                        const double* dT_M, int n, int max_step, int N, int nm, const int* ls, const int* ms, const double* nqc,
                        const double* rd, const double* binf, const int* bini, double* hplus, double* hcross, int* nsamp, void* stream) {
    ImrModes mm;
    int rc = make_modes(mm, nm, ls, ms);
    if (rc) return rc;
    EOBHIP_REQUIRE(n >= 0 && n <= 65535 && N >= 1, "bad sizes");
    if (n == 0) return EOBHIP_OK;
    ResampleShape s = resample_shape(N, n, kImrRoom);
    s.grid.x += kRingBlocks;
    hipLaunchKernelGGL(s.rows == 1 ? k_imr_resample<1> : k_imr_resample<kRunRows>, s.grid, s.block, s.lds, as_stream(stream), dense,
                       num_steps, coef, rp_coef, amp, dT_M, max_step, N, nm, mode_order(mm.m, nm), nqc, rd, binf, bini, hplus, hcross, nsamp);
    return check_launch("imr_resample");
}

size_t eobhip_imr_rd_doubles(void) { return kRdCount; }
size_t eobhip_imr_bin_doubles(void) { return kBinCount; }
size_t eobhip_imr_bin_ints(void) { return kBinICount; }

}  // extern "C"
