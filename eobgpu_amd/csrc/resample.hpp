// Uniform resampling of splines by wavefronts.
//
// A wavefront takes a run of consecutive samples t_j of one binary, 128 at a
// time (two per lane, one 16-byte store per series), and keeps the knot
// interval (searchsorted(t, t_j, 'right') - 1, eob/seobnrv4phm.py:241-272) it is
// in.  Most rows of 128 lie in one interval: the row's last time against the next
// knot decides that with one comparison, and the interval's coefficients are then
// read once for the wavefront through the scalar cache.  A row that passes knots
// reads up to 64 of them, one per lane, and each lane counts those at or before
// its samples; only a row that passes many falls back to a bisection per
// sample.  No LDS, no barriers: what a block waited for before (a window of
// knots staged for 4096 samples, then a bisection of it per sample) was most of
// these kernels' time.
#pragma once
#include <hip/hip_runtime.h>

#include "eob_fastmath.hpp"

namespace eobhip_detail {

constexpr int kRow = 128;                 // samples per wavefront and step
constexpr int kRunRows = 8;               // rows of a run
constexpr int kFewKnots = 8;              // knots a row may pass before its lanes bisect
constexpr int kRun = kRow * kRunRows;     // samples per run

// sin and cos of x: x - n pi/2 in two fused steps (the first exact for |n| <
// 2^20), the Taylor series through r^17 and r^16 on |r| <= pi/4 (first omitted
// terms below 2e-18), and the quadrant; the library's for larger x anywhere in
// the wavefront.  Within 1e-16 absolute of it; the arguments here are phases of
// 10 to 10^4 rad whose own rounding is 1e-15 to 1e-12.  About 40 instructions
// against the library's 75.
__device__ __forceinline__ void sincos_phase(double x, double* s, double* c) {
    if (__any(!(fabs(x) < 1.0e6))) {
        sincos(x, s, c);
        return;
    }
    constexpr double kTwoOverPi = 0x1.45f306dc9c883p-1, kPio2Hi = 0x1.921fb54442d18p+0, kPio2Lo = 0x1.1a62633145c07p-54;
    const double n = rint(x * kTwoOverPi);
    const double r = fma(-n, kPio2Lo, fma(-n, kPio2Hi, x));
    const double z = r * r;
    double p = fma(z, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
    p = fma(p, z, 1.0 / 6227020800.0);
    p = fma(p, z, -1.0 / 39916800.0);
    p = fma(p, z, 1.0 / 362880.0);
    p = fma(p, z, -1.0 / 5040.0);
    p = fma(p, z, 1.0 / 120.0);
    p = fma(p, z, -1.0 / 6.0);
    const double sr = fma(r * z, p, r);
    double q = fma(z, 1.0 / 20922789888000.0, -1.0 / 87178291200.0);
    q = fma(q, z, 1.0 / 479001600.0);
    q = fma(q, z, -1.0 / 3628800.0);
    q = fma(q, z, 1.0 / 40320.0);
    q = fma(q, z, -1.0 / 720.0);
    q = fma(q, z, 1.0 / 24.0);
    q = fma(q, z, -0.5);
    const double cr = fma(q, z, 1.0);
    const int k = (int)n;
    const double a = (k & 1) ? cr : sr, b = (k & 1) ? sr : cr;
    *s = (k & 2) ? -a : a;
    *c = ((k + 1) & 2) ? -b : b;
}

// searchsorted(T, t, 'right') - 1, at least 0, for a wavefront-uniform t: 64
// knots are compared at once.  T: knot times at stride 5, sorted, len >= 1.
__device__ __forceinline__ int wave_interval(const double* __restrict__ T, int len, double t) {
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = len;   // knots before lo are <= t, knots from hi on are > t
    while (hi - lo > 64) {
        const int step = (hi - lo + 63) >> 6;
        const int k = lo + lane * step;
        const int c = __popcll(__ballot(k < hi && T[5 * (size_t)(k < hi ? k : hi - 1)] <= t));
        if (c == 0) {
            hi = lo;
            break;
        }
        hi = lo + c * step < hi ? lo + c * step : hi;
        lo = lo + (c - 1) * step + 1;
    }
    if (hi > lo) {
        const int k = lo + lane;
        lo += __popcll(__ballot(k < hi && T[5 * (size_t)(k < hi ? k : hi - 1)] <= t));
    }
    return lo > 0 ? lo - 1 : 0;
}

// lane q's value, q uniform
__device__ __forceinline__ double lane_value(double v, int q) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), q), hi = __builtin_amdgcn_readlane((int)(b >> 32), q);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

typedef const __attribute__((address_space(4))) double* ConstPtr;

// The rows of the run that starts at sample j0, as far as samples have a value
// (j < jend; j0 < jend):
//   time(j)                       the time of sample j
//   enter(i)                      the wavefront is in interval i from here on (uniform)
//   one(j, ta, tb, full)          a row in that interval: samples j, j + 1 of this lane;
//                                 full: all of the row's samples are below jend
//   each(j, ta, tb, ia, ib)       a row that passes knots: each sample's own interval
// kLastApart: rows past the last knot go to each as well (its interval has a value
// and no slope there).
template <bool kLastApart = false, class Time, class Enter, class One, class Each>
__device__ __forceinline__ void resample_rows(const double* __restrict__ T, int len, long long j0, long long jend, const Time& time,
                                              const Enter& enter, const One& one, const Each& each) {
    const int lane = threadIdx.x & 63;
    int ind = wave_interval(T, len, time(j0));
    for (int r = 0; r < kRunRows;) {
        if (j0 + (long long)r * kRow >= jend) break;
        const double next = ind + 1 < len ? ((ConstPtr)T)[5 * (size_t)(ind + 1)] : (kLastApart ? -HUGE_VAL : HUGE_VAL);
        enter(ind);
        double last = 0.0;
        for (; r < kRunRows; ++r) {
            const long long jr = j0 + (long long)r * kRow;
            if (jr >= jend) return;
            const bool full = jr + kRow <= jend;
            last = time(full ? jr + kRow - 1 : jend - 1);
            if (!__builtin_amdgcn_readfirstlane(last < next)) break;
            const long long j = jr + 2 * lane;
            one(j, time(j), time(j + 1), full);
        }
        if (r == kRunRows) break;
        const long long j = j0 + (long long)r * kRow + 2 * lane;
        const double ta = time(j), tb = time(j + 1);
        const int k = ind + 1 + lane;
        const double tk = k < len ? T[5 * (size_t)k] : HUGE_VAL;
        const int passed = __popcll(__ballot(tk <= last));
        int ia = ind, ib = ind;
        if (passed <= kFewKnots) {
            for (int q = 0; q < passed; ++q) {
                const double x = lane_value(tk, q);
                ia += x <= ta;
                ib += x <= tb;
            }
            ind += passed;
        } else {
            // T[ind] <= every sample of the row (or ind = 0)
            for (int m = len - ind; m > 1;) {
                const int half = m >> 1;
                ia = T[5 * (size_t)(ia + half)] <= ta ? ia + half : ia;
                ib = T[5 * (size_t)(ib + half)] <= tb ? ib + half : ib;
                m -= half;
            }
            ind = passed < 64 ? ind + passed : wave_interval(T, len, last);
        }
        each(j, ta, tb, ia, ib);
        ++r;
    }
}

// A lane's two samples in turn, f(t, i, re, im) each: where a wavefront gathers
// rows per lane, two samples' at once would double the registers of the whole
// kernel.
template <class F>
__device__ __forceinline__ void one_by_one(double ta, double tb, int ia, int ib, double (&re)[2], double (&im)[2], const F& f) {
#pragma unroll 1
    for (int e = 0; e < 2; ++e) {
        double x, y;
        f(e ? tb : ta, e ? ib : ia, x, y);
        re[0] = e ? re[0] : x;
        im[0] = e ? im[0] : y;
        re[1] = x;
        im[1] = y;
    }
}

// Two consecutive samples of a series of N.  kStream: past the caches (a series
// longer than they hold: 1682 us for the five-mode sum of 512 binaries x 2^20
// against 2496 through them).
typedef double SamplePair __attribute__((ext_vector_type(2), aligned(8)));
template <bool kStream>
__device__ __forceinline__ void store_pair(double* out, long long j, long long N, double a, double b) {
    if (j + 1 < N) {
        SamplePair v = {a, b};
        if constexpr (kStream) __builtin_nontemporal_store(v, reinterpret_cast<SamplePair*>(out + j));
        else *reinterpret_cast<SamplePair*>(out + j) = v;
    } else if (j < N) {
        out[j] = a;
    }
}

// h22 = S e^{-2 i phi} at x past the knot of a row of the (2,2) splines (phi,
// Re S, Im S; 4 coefficients each)
template <class Row>
__device__ __forceinline__ void h22_sample(const Row& c, double x, double& re, double& im) {
    const double x2 = x * x, x3 = x2 * x;
    const double ph = c[0] + c[1] * x + c[2] * x2 + c[3] * x3;
    const double sr = c[4] + c[5] * x + c[6] * x2 + c[7] * x3;
    const double si = c[8] + c[9] * x + c[10] * x2 + c[11] * x3;
    double sp, cp;
    sincos_phase(2.0 * ph, &sp, &cp);
    re = sr * cp + si * sp;
    im = si * cp - sr * sp;
}

// one interval's row of them and its knot, through the scalar cache (the tables
// are read-only while the kernels run)
struct H22Row {
    double c[12], tk;
    __device__ __forceinline__ void load(const double* T, const double* C, int i) {
        const ConstPtr r = (ConstPtr)(C + (size_t)12 * i);
#pragma unroll
        for (int q = 0; q < 12; ++q) c[q] = r[q];
        tk = ((ConstPtr)T)[5 * (size_t)i];
    }
};

// h22 on the run of samples t0 + j dT from j0: put(j, re[2], im[2], full)
template <class Put>
__device__ __forceinline__ void h22_rows(const double* __restrict__ T, const double* __restrict__ C, int len, double t0, double dT, long long j0,
                                         long long jend, const Put& put) {
    H22Row row;
    resample_rows(
        T, len, j0, jend, [&](long long j) { return t0 + (double)j * dT; }, [&](int i) { row.load(T, C, i); },
        [&](long long j, double ta, double tb, bool full) {
            double re[2], im[2];
            h22_sample(row.c, ta - row.tk, re[0], im[0]);
            h22_sample(row.c, tb - row.tk, re[1], im[1]);
            put(j, re, im, full);
        },
        [&](long long j, double ta, double tb, int ia, int ib) {
            double re[2], im[2];
            one_by_one(ta, tb, ia, ib, re, im, [&](double t, int i, double& x, double& y) { h22_sample(C + (size_t)12 * i, t - T[5 * (size_t)i], x, y); });
            put(j, re, im, false);
        });
}

// h+ and hx (hx may be null) of N samples, zero from nb on
struct SeriesOut {
    double *out, *outc;
    double a;
    long long nb, N;
    __device__ __forceinline__ void put(long long j, const double (&re)[2], const double (&im)[2], bool full) const {
        const bool va = full || j < nb, vb = full || j + 1 < nb;
        store_pair<true>(out, j, N, va ? a * re[0] : 0.0, vb ? a * re[1] : 0.0);
        if (outc) store_pair<true>(outc, j, N, va ? a * im[0] : 0.0, vb ? a * im[1] : 0.0);
    }
    // the run's rows without a sample below nb
    __device__ __forceinline__ void zeros(long long j0) const {
        const long long k = nb > j0 ? (nb - j0 + kRow - 1) / kRow : 0;
        for (int r = k < kRunRows ? (int)k : kRunRows; r < kRunRows; ++r) {
            const long long j = j0 + (long long)r * kRow + 2 * (threadIdx.x & 63);
            store_pair<true>(out, j, N, 0.0, 0.0);
            if (outc) store_pair<true>(outc, j, N, 0.0, 0.0);
        }
    }
};

// A wavefront's runs of one binary's series (grid.x blocks of `waves` wavefronts): f(j0)
template <class F>
__device__ __forceinline__ void for_runs(long long N, int waves, const F& f) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long nrun = (N + kRun - 1) / kRun;
    for (long long run = (long long)blockIdx.x * waves + wave; run < nrun; run += (long long)gridDim.x * waves) f(run * kRun);
}

// Blocks (of four wavefronts) per binary: about 16384 in all (64 per CU), no
// more, so that a wavefront takes several runs.  They are spread over the series
// (run, run + the binary's wavefronts, ...), since the template's part costs more
// than the zeros after it.  h+ of 256 binaries x 2^20 and the five-mode sum of
// 512: a block per 4096 samples 540 and 2499 us, 16384 blocks 468 and 1682, 4096
// blocks 501 and 1746; contiguous runs per block 772 and 3510.
inline int resample_blocks(int N, int n) {
    const int most = (int)((N + 4LL * kRun - 1) / (4LL * kRun)), want = (16384 + n - 1) / n;
    return want < most ? want : most;
}

// The modes of a sum by falling m: mode q[k] is the k-th, down[k] = m[q[k-1]] -
// m[q[k]] (0 for k = 0), down[nm] the last one's m.
constexpr int kMaxModes = 15;
struct ModeOrder {
    int q[kMaxModes], down[kMaxModes + 1];
};
inline ModeOrder mode_order(const int* m, int nm) {
    ModeOrder o{};
    for (int k = 0; k < nm; ++k) {
        int j = k;
        for (; j > 0 && m[o.q[j - 1]] < m[k]; --j) o.q[j] = o.q[j - 1];
        o.q[j] = k;
    }
    for (int k = 1; k < nm; ++k) o.down[k] = m[o.q[k - 1]] - m[o.q[k]];
    o.down[nm] = m[o.q[nm - 1]];
    return o;
}

}  // namespace eobhip_detail
