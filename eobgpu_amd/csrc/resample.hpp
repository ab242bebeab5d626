// Uniform resampling of splines by wavefronts.
//
// A wavefront takes a run of consecutive samples t_j of one binary, 128 at a
// time (two per lane, one 16-byte store per series), and keeps the knot
// interval (searchsorted(t, t_j, 'right') - 1, eob/seobnrv4phm.py:241-272) it is
// in.  Most rows of 128 lie in one interval: the row's last time against the next
// knot decides that with one comparison.  The run's knots and table rows are
// staged at its start, by and for the wavefront alone (no barriers).
#pragma once
#include <hip/hip_runtime.h>

#include "eob_fastmath.hpp"

namespace eobhip_detail {

constexpr int kRow = 128;                 // samples per wavefront and step
constexpr int kRunRows = 4;               // rows of a run
constexpr int kRun = kRow * kRunRows;     // samples per run

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

// two consecutive doubles at any 8-byte boundary
typedef double SamplePair __attribute__((ext_vector_type(2), aligned(8)));

// A lane's two samples in turn, f(i, x, re, im) each: at once they would double the
// registers of the whole kernel.  Whether f was true for both.
template <class F>
__device__ __forceinline__ bool one_by_one(double xa, double xb, int ia, int ib, double (&re)[2], double (&im)[2], const F& f) {
    bool good = true;
#pragma unroll 1
    for (int e = 0; e < 2; ++e) {
        double x, y;
        good &= f(e ? ib : ia, e ? xb : xa, x, y);
        re[0] = e ? re[0] : x;
        im[0] = e ? im[0] : y;
        re[1] = x;
        im[1] = y;
    }
    return good;
}

// How a sample's sine and cosine are taken: kBounded only for |x| < 2^49 (false for the
// others), kAny for any.  Rows are taken by the first and once more by the second if a
// phase of theirs is larger: with the large reduction inside the loops the likelihood of
// 1024 templates takes 5% longer, that of 512 with 5k to 60k knots 3%.
enum Phases { kBounded, kAny };
template <Phases P>
__device__ __forceinline__ bool sincos_of(double x, double& s, double& c) {
    if constexpr (P == kBounded) return eob::sincos_bounded(x, s, c);
    eob::sincos_phase(x, s, c);
    return true;
}

// A wavefront's LDS copy of R consecutive rows of a table, CS doubles each
template <int CS, int R>
struct StagedRows {
    static constexpr int kRows = R;
    __attribute__((aligned(16))) double c[R * CS];
    // n <= R rows of `cs` <= CS doubles from src on
    __device__ __forceinline__ void copy(const double* __restrict__ src, int n, int cs = CS) {
        constexpr int kSteps = (R * CS + 127) / 128;
        const int lane = threadIdx.x & 63;
        SamplePair v[kSteps];
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int i = 2 * (lane + 64 * q);
            if (i < n * cs) v[q] = *reinterpret_cast<const SamplePair*>(src + i);
        }
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int i = 2 * (lane + 64 * q);
            if (i < n * cs) *reinterpret_cast<double2*>(c + i) = make_double2(v[q].x, v[q].y);
        }
    }
    __device__ __forceinline__ const double* row(int k) const { return c + k * CS; }
    // row k of 4-coefficient series keeps its values and loses its slopes
    __device__ __forceinline__ void flatten(int k, int cs = CS) {
        for (int i = threadIdx.x & 63; i < cs; i += 64)
            if (i & 3) c[k * cs + i] = 0.0;
    }
};

// The rows of the run that starts at sample j0, as far as samples have a value
// (j < jend; j0 < jend):
//   time(j)                the time of sample j
//   stage(i, n)            table rows i .. i + n - 1 (n <= R) into the wavefront's LDS
//   near(k, x, re, im)     one sample at x past the knot of staged row k (per lane); false
//                          if its phase needs `exact`
//   far(i, x, re, im)      the same from table row i (per lane), read from memory
//   exact(i, x, re, im)    the same for any phase
//   put(j, re, im, full)   a lane's samples j, j + 1 (full: all of the row's are below jend)
// The run's knots (lane q holds the q-th after its first) and table rows are read
// in two steps at its start; its rows then wait for no load.  Interval by interval
// through the scalar cache, with gathers where a row passes a knot, the waits
// (about 1 us each, four a row) were the time: 1024 templates' h+ for the likelihood
// 880 us, 735 this way; the five modes with NQC factors of 512 binaries 3560, 3060.
template <int R, class Time, class Stage, class Near, class Far, class Exact, class Put>
__device__ __forceinline__ void resample_rows(const double* __restrict__ T, int len, long long j0, long long jend, const Time& time,
                                              const Stage& stage, const Near& near, const Far& far, const Exact& exact, const Put& put) {
    static_assert(R <= 63, "a lane per knot");
    const int lane = threadIdx.x & 63;
    const double end = time((j0 + kRun < jend ? j0 + kRun : jend) - 1);
    int ind = wave_interval(T, len, time(j0));
    for (int r = 0; r < kRunRows;) {
        if (j0 + (long long)r * kRow >= jend) break;
        // staged: rows ind .. ind + cnt, local 0 .. cnt
        const int kl = ind + 1 + lane;
        const double tk = kl < len ? T[5 * (size_t)kl] : HUGE_VAL;
        double t0 = ((ConstPtr)T)[5 * (size_t)ind];   // the current interval's knot
        int cnt = __popcll(__ballot(kl < len && tk <= end));
        cnt = cnt < R ? cnt : R - 1;
        stage(ind, cnt + 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int cur = 0;
        double next = lane_value(tk, 0), last = 0.0;
        long long j = 0;
        double re[2], im[2];
        bool covered = true, large = false;
        for (; r < kRunRows; ++r) {
            const long long jr = j0 + (long long)r * kRow;
            if (jr >= jend) return;
            const bool full = jr + kRow <= jend;
            j = jr + 2 * lane;
            last = time(full ? jr + kRow - 1 : jend - 1);
            const double ta = time(j), tb = time(j + 1);
            int ia = cur, ib = cur;
            double xa = t0, xb = t0;
            if (!__builtin_amdgcn_readfirstlane(last < next)) {
                const int to = __popcll(__ballot(tk <= last));
                covered = to <= cnt;
                if (!covered) break;
                for (; cur < to; ++cur) {
                    t0 = lane_value(tk, cur);
                    ia = t0 <= ta ? cur + 1 : ia;
                    ib = t0 <= tb ? cur + 1 : ib;
                    xa = t0 <= ta ? t0 : xa;
                    xb = t0 <= tb ? t0 : xb;
                }
                next = lane_value(tk, cur);
            }
            large = __any(!one_by_one(ta - xa, tb - xb, ia, ib, re, im, near));
            if (large) break;
            put(j, re, im, full);
        }
        if (covered && !large) break;
        if (!large && cur > 0) {   // stage from here
            ind += cur;
            continue;
        }
        // the row passes more knots than are staged, or has a phase that near leaves out: T[ind]
        // <= every sample of it (or ind = 0)
        const double ta = time(j), tb = time(j + 1);
        int ia = ind, ib = ind;
        for (int m = len - ind; m > 1;) {
            const int half = m >> 1;
            ia = T[5 * (size_t)(ia + half)] <= ta ? ia + half : ia;
            ib = T[5 * (size_t)(ib + half)] <= tb ? ib + half : ib;
            m -= half;
        }
        const double xa = ta - T[5 * (size_t)ia], xb = tb - T[5 * (size_t)ib];
        if (!large) large = __any(!one_by_one(xa, xb, ia, ib, re, im, far));
        if (large) one_by_one(xa, xb, ia, ib, re, im, exact);
        put(j, re, im, false);
        ind = wave_interval(T, len, last);
        ++r;
    }
}

// Two consecutive samples of a series of N.  kStream: past the caches.  The mode sum
// of 512 binaries x 2^20 1682 us against 2496 through them, h+ of 64 x 2^18 46 against
// 50, of one binary the same; what reads the series next loses at most what that
// gains (h+ and its transform, streamed and not: 256 x 2^20 2183 and 2204 us, 64 x
// 2^17 85 and 76, 16 x 2^14 20 and 20, 1 x 2^20 30 and 29), so that no size is worth a rule.
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
template <Phases P, class Row>
__device__ __forceinline__ bool h22_sample(const Row& c, double x, double& re, double& im) {
    const double x2 = x * x, x3 = x2 * x;
    const double ph = c[0] + c[1] * x + c[2] * x2 + c[3] * x3;
    const double sr = c[4] + c[5] * x + c[6] * x2 + c[7] * x3;
    const double si = c[8] + c[9] * x + c[10] * x2 + c[11] * x3;
    double sp, cp;
    const bool good = sincos_of<P>(2.0 * ph, sp, cp);
    re = sr * cp + si * sp;
    im = si * cp - sr * sp;
    return good;
}

// h22 on the run of samples t0 + j dT from j0: put(j, re[2], im[2], full)
typedef StagedRows<12, 16> H22Stage;
template <class Put>
__device__ __forceinline__ void h22_rows(H22Stage& st, const double* __restrict__ T, const double* __restrict__ C, int len, double t0, double dT,
                                         long long j0, long long jend, const Put& put) {
    resample_rows<H22Stage::kRows>(
        T, len, j0, jend, [&](long long j) { return t0 + (double)j * dT; }, [&](int i, int n) { st.copy(C + (size_t)12 * i, n); },
        [&](int k, double x, double& re, double& im) { return h22_sample<kBounded>(st.row(k), x, re, im); },
        [&](int i, double x, double& re, double& im) { return h22_sample<kBounded>(C + (size_t)12 * i, x, re, im); },
        [&](int i, double x, double& re, double& im) { return h22_sample<kAny>(C + (size_t)12 * i, x, re, im); }, put);
}

// h+ and hx (hx may be null) of N samples, zero from nb on.  kHole: but samples nb <= j <
// hole are left as they are.
template <bool kHole = false>
struct SeriesOut {
    double *out, *outc;
    double a;
    long long nb, N, hole = 0;
    __device__ __forceinline__ void pair(double* o, long long j, double x, double y) const {
        if (!kHole || j + 1 < nb || j >= hole) {
            store_pair<true>(o, j, N, x, y);
        } else {
            if (j < nb && j < N) o[j] = x;
            if (j + 1 >= hole && j + 1 < N) o[j + 1] = y;
        }
    }
    __device__ __forceinline__ void put(long long j, const double (&re)[2], const double (&im)[2], bool full) const {
        const bool va = full || j < nb, vb = full || j + 1 < nb;
        pair(out, j, va ? a * re[0] : 0.0, vb ? a * re[1] : 0.0);
        if (outc) pair(outc, j, va ? a * im[0] : 0.0, vb ? a * im[1] : 0.0);
    }
    // the run's rows without a sample below nb
    __device__ __forceinline__ void zeros(long long j0) const {
        const long long k = nb > j0 ? (nb - j0 + kRow - 1) / kRow : 0;
        for (int r = k < kRunRows ? (int)k : kRunRows; r < kRunRows; ++r) {
            const long long j = j0 + (long long)r * kRow + 2 * (threadIdx.x & 63);
            pair(out, j, 0.0, 0.0);
            if (outc) pair(outc, j, 0.0, 0.0);
        }
    }
};

// A wavefront's runs of one binary's series by `blocks` blocks, f(j0); grid resample_grid
template <class F>
__device__ __forceinline__ void for_runs(long long N, int waves, unsigned blocks, const F& f) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long nrun = (N + kRun - 1) / kRun;
    for (long long run = (long long)blockIdx.x * waves + wave; run < nrun; run += (long long)blocks * waves) f(run * kRun);
}

// (blocks of four wavefronts, binaries): about 131072 blocks in all, no more, so
// that a wavefront takes several runs.  They are spread over the series (run, run +
// the binary's wavefronts, ...), since the template's part costs more than the
// zeros after it.  h+ of 256 binaries x 2^20, the five-mode sum of 512 and the same
// with its ringdown at 16384 Hz: 16384 blocks of runs of 8 rows 461, 1675 and 3165
// us, 131072 of 4 rows 407, 1620 and 2990, 524288 409, 1581 and 3076; neighbouring
// blocks on different binaries instead 480, 1690 and 3700 (writes all over
// memory), contiguous runs per block slower by half.
inline dim3 resample_grid(int N, int n) {
    const int most = (int)((N + 4LL * kRun - 1) / (4LL * kRun)), want = (131072 + n - 1) / n;
    return dim3(want < most ? want : most, n);
}

constexpr int kMaxModes = 15;

// The modes of a sum by falling m, four bits each (two scalar registers a list,
// where arrays would be loaded entry by entry): q(k) the k-th mode, down(k) =
// m[q(k-1)] - m[q(k)] (0 for k = 0), down(nm) the last one's m.
struct ModeOrder {
    unsigned long long qs = 0, downs = 0;
    __device__ __forceinline__ int q(int k) const { return (int)(qs >> (4 * k)) & 15; }
    __device__ __forceinline__ int down(int k) const { return (int)(downs >> (4 * k)) & 15; }
};
inline ModeOrder mode_order(const int* m, int nm) {   // nm <= 15, 1 <= m <= 15
    int q[16];
    for (int k = 0; k < nm; ++k) {
        int j = k;
        for (; j > 0 && m[q[j - 1]] < m[k]; --j) q[j] = q[j - 1];
        q[j] = k;
    }
    ModeOrder o;
    for (int k = 0; k < nm; ++k) {
        o.qs |= (unsigned long long)q[k] << (4 * k);
        o.downs |= (unsigned long long)(m[q[k]] - (k + 1 < nm ? m[q[k + 1]] : 0)) << (4 * (k + 1));
    }
    return o;
}

}  // namespace eobhip_detail
