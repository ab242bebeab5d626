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
constexpr int kRunRows = 4;               // most rows of a run
constexpr int kRun = kRow * kRunRows;

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

// the wavefront's number in its block
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

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

// From a row's samples lane, 64 + lane to its samples 2 lane, 2 lane + 1
__device__ __forceinline__ void pairs_of(double (&v)[2]) {
    const int lane = threadIdx.x & 63, from = 2 * lane & 63;
    const double a0 = __shfl(v[0], from), a1 = __shfl(v[0], from + 1), b0 = __shfl(v[1], from), b1 = __shfl(v[1], from + 1);
    v[0] = lane < 32 ? a0 : b0;
    v[1] = lane < 32 ? a1 : b1;
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

// A wavefront's LDS copy of n consecutive rows of a table, cs (even) doubles each; c at
// 16 bytes.  128 kSteps doubles are on their way at once.
template <int kSteps>
__device__ __forceinline__ void stage_rows(double* c, const double* __restrict__ src, int n, int cs) {
    for (int i0 = 2 * (threadIdx.x & 63); i0 < n * cs; i0 += 128 * kSteps) {
        SamplePair v[kSteps];
#pragma unroll
        for (int q = 0; q < kSteps; ++q)
            if (i0 + 128 * q < n * cs) v[q] = *reinterpret_cast<const SamplePair*>(src + i0 + 128 * q);
#pragma unroll
        for (int q = 0; q < kSteps; ++q)
            if (i0 + 128 * q < n * cs) *reinterpret_cast<double2*>(c + i0 + 128 * q) = make_double2(v[q].x, v[q].y);
    }
}

// A staged row of 4-coefficient series keeps its values and loses its slopes
__device__ __forceinline__ void flatten_row(double* c, int cs) {
    for (int i = threadIdx.x & 63; i < cs; i += 64)
        if (i & 3) c[i] = 0.0;
}

// How many rows of cs doubles are staged at once in `room` doubles: with them, at most
// 62 knots after the first, whose times the lanes hold
constexpr int kMostStaged = 63;
__device__ __forceinline__ int staged_rows(int room, int cs) { return room / cs < kMostStaged ? room / cs : kMostStaged; }

// The `rows` rows of the run that starts at sample j0, as far as samples have a value
// (j < jend; j0 < jend), R table rows staged at once:
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
//
// R is what fits in the LDS that the kernel's wavefronts have anyway: tables of 16384
// binaries with 17 knots a row of 128 samples take 579 us with R = 63 where one by one
// (2, 2) rows of 16 go to memory (1197), 603 and 1073 with one and five modes (1288 and
// 2286 with 8 rows).  A row that passes R knots or more is read from memory, by
// lane l its samples l and 64 + l, whose table rows are neighbours (2 l and 2 l + 1
// touch every line twice: 224 us for 129 with 60 knots a row and five modes), its knots
// from the lanes for as many rows as they cover (keep; without, the likelihood's
// kernel spills less, and its rows pass fewer).
template <class Time, class Stage, class Near, class Far, class Exact, class Put>
__device__ __forceinline__ void resample_rows(int rows, int R, bool keep, const double* __restrict__ T, int len, long long j0,
                                              long long jend, const Time& time,
                                              const Stage& stage, const Near& near, const Far& far, const Exact& exact, const Put& put) {
    const int lane = threadIdx.x & 63;
    const double end = time((j0 + rows * kRow < jend ? j0 + rows * kRow : jend) - 1);
    int ind = wave_interval(T, len, time(j0));
    bool large = false;   // the next row needs `exact`
    for (int r = 0; r < rows;) {
        const long long jr0 = j0 + (long long)r * kRow;
        if (jr0 >= jend) break;
        const int kl = ind + 1 + lane;
        const double tk = kl < len ? T[5 * (size_t)kl] : __builtin_nan("");   // past no time
        double t0 = ((ConstPtr)T)[5 * (size_t)ind];   // the current interval's knot
        double re[2], im[2];
        // samples ta, tb to the intervals after the knots from .. to - 1 (of the 64 of tk)
        const auto pass = [&](int from, int to, double ta, double tb, int& ia, int& ib, double& xa, double& xb) {
            for (int q = from; q < to; ++q) {
                t0 = lane_value(tk, q);
                ia = t0 <= ta ? q + 1 : ia;
                ib = t0 <= tb ? q + 1 : ib;
                xa = t0 <= ta ? t0 : xa;
                xb = t0 <= tb ? t0 : xb;
            }
        };
        const bool full0 = jr0 + kRow <= jend;
        const double last0 = time(full0 ? jr0 + kRow - 1 : jend - 1);
        const int first = __popcll(__ballot(tk <= last0));   // knots that the next row passes (64: or more)
        if (__builtin_expect(first >= R || large, 0)) {
            // rows that pass more than can be staged, or have a phase that near leaves out: from memory
            int cur = 0, to = first;
            long long jr = jr0;
            double last = last0;
            do {
                const bool full = jr + kRow <= jend;
                const double ta = time(jr + lane), tb = time(jr + 64 + lane);
                int ia = cur, ib = cur;
                double xa = t0, xb = t0;
                if (to < 64) {
                    pass(cur, to, ta, tb, ia, ib, xa, xb);
                    ia += ind;
                    ib += ind;
                } else {   // T[ind] <= every sample of the row (or ind = 0)
                    ia = ib = ind;
                    for (int m = len - ind; m > 1;) {
                        const int half = m >> 1;
                        ia = T[5 * (size_t)(ia + half)] <= ta ? ia + half : ia;
                        ib = T[5 * (size_t)(ib + half)] <= tb ? ib + half : ib;
                        m -= half;
                    }
                    xa = T[5 * (size_t)ia];
                    xb = T[5 * (size_t)ib];
                }
                if (!large) large = __any(!one_by_one(ta - xa, tb - xb, ia, ib, re, im, far));
                if (large) one_by_one(ta - xa, tb - xb, ia, ib, re, im, exact);
                large = false;
                pairs_of(re);
                pairs_of(im);
                put(jr + 2 * lane, re, im, full);
                ++r;
                cur = to;
                jr += kRow;
                if (!keep || cur >= 64 || r == rows || jr >= jend) break;
                last = time(jr + kRow <= jend ? jr + kRow - 1 : jend - 1);
                to = __popcll(__ballot(tk <= last));
            } while (to < 64 && to - cur >= R);
            ind = cur < 64 ? ind + cur : wave_interval(T, len, last);
            continue;
        }
        // staged: rows ind .. ind + cnt, local 0 .. cnt
        int cnt = __popcll(__ballot(tk <= end));
        cnt = cnt < R ? cnt : R - 1;
        stage(ind, cnt + 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int cur = 0, to = first;
        double next = lane_value(tk, to);
        for (long long jr = jr0;;) {
            const bool full = jr + kRow <= jend;
            const long long j = jr + 2 * lane;
            const double ta = time(j), tb = time(j + 1);
            int ia = cur, ib = cur;
            double xa = t0, xb = t0;
            pass(cur, to, ta, tb, ia, ib, xa, xb);
            large = __any(!one_by_one(ta - xa, tb - xb, ia, ib, re, im, near));
            if (large) break;
            put(j, re, im, full);
            cur = to;
            jr += kRow;
            if (++r == rows || jr >= jend) return;
            const double last = time(jr + kRow <= jend ? jr + kRow - 1 : jend - 1);
            if (!__builtin_amdgcn_readfirstlane(last < next)) {
                to = __popcll(__ballot(tk <= last));
                if (to > cnt) break;
                next = lane_value(tk, to);
            }
        }
        ind += cur;   // stage from here
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

// h22 on the run of samples t0 + j dT from j0: put(j, re[2], im[2], full).  st: 12 R doubles of LDS
template <class Put>
__device__ __forceinline__ void h22_rows(double* st, int rows, int R, bool keep, const double* __restrict__ T, const double* __restrict__ C,
                                         int len, double t0, double dT, long long j0, long long jend, const Put& put) {
    resample_rows(
        rows, R, keep, T, len, j0, jend, [&](long long j) { return t0 + (double)j * dT; },
        [&](int i, int n) { stage_rows<2>(st, C + (size_t)12 * i, n, 12); },
        [&](int k, double x, double& re, double& im) { return h22_sample<kBounded>(st + 12 * k, x, re, im); },
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
    __device__ __forceinline__ void zeros(long long j0, int rows) const {
        const long long k = nb > j0 ? (nb - j0 + kRow - 1) / kRow : 0;
#pragma unroll
        for (int r = 0; r < kRunRows; ++r) {
            if (r < k || r >= rows) continue;
            const long long j = j0 + (long long)r * kRow + 2 * (threadIdx.x & 63);
            pair(out, j, 0.0, 0.0);
            if (outc) pair(outc, j, 0.0, 0.0);
        }
    }
};

// A wavefront's runs of `rows` rows of one binary's series by `blocks` blocks, of which its
// is number `block`, f(j0); shape resample_shape
template <class F>
__device__ __forceinline__ void for_runs(long long N, int rows, unsigned block, unsigned blocks, const F& f) {
    const long long step = (long long)blocks * (blockDim.x >> 6) * (rows * kRow);
    for (long long j0 = ((long long)block * (blockDim.x >> 6) + wave_index()) * (rows * kRow); j0 < N; j0 += step) f(j0);
}

// (blocks of up to four wavefronts, binaries): about 131072 blocks in all, no more, so
// that a wavefront takes several runs.  They are spread over the series (run, run +
// the binary's wavefronts, ...), since the template's part costs more than the
// zeros after it.  h+ of 256 binaries x 2^20, the five-mode sum of 512 and the same
// with its ringdown at 16384 Hz: 16384 blocks of runs of 8 rows 461, 1675 and 3165
// us, 131072 of 4 rows 407, 1620 and 2990, 524288 409, 1581 and 3076; neighbouring
// blocks on different binaries instead 480, 1690 and 3700 (writes all over
// memory), contiguous runs per block slower by half.
//
// Runs of one row while all rows together are fewer than two a SIMD of four wavefronts
// (8192): a run's rows wait for each other, and there is room.  Merger-ringdown
// templates of five modes, 1 binary x 2^16 and 64 x 2^12: 20.2 and 23.7 us with runs of
// four, 8.3 and 13.0; 512 binaries x 2048 with 250 knots a row (8192 rows) 62.0 with
// four, 71.1 with one; 4 x 2^18 (8192 rows) 17.4 and 20.1.  No more wavefronts in a
// block than there are runs: each has its LDS whether it has a run or not (65535
// binaries x 256 samples, one mode, 134 us; 398 with four).
struct ResampleShape {
    dim3 grid, block;
    size_t lds;
    int rows;   // of a run
};
constexpr int kFewRows = 8192;
inline ResampleShape resample_shape(int N, int n, int room) {   // room: doubles staged by a wavefront
    const int rows = (long long)n * ((N + (long long)kRow - 1) / kRow) < kFewRows ? 1 : kRunRows;
    const long long runs = (N + (long long)rows * kRow - 1) / (rows * kRow);
    const int waves = runs < 4 ? (int)runs : 4, most = (int)((runs + waves - 1) / waves), want = (131072 + n - 1) / n;
    return {dim3(want < most ? want : most, n), dim3(64 * waves), sizeof(double) * room * waves, rows};
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
