// Batched not-a-knot cubic splines, uniform resampling of the (2,2) mode, the
// real-to-complex FFT of the templates and the frequency-domain likelihood.
//
// Reference: interpolate_TD (src/interpolate.cu:11-308), CubicSplineInterpolantTD
// (eob/seobnrv4phm.py:161-386), compute_full_waveform's resampling of
// h_lm e^{i m phi} and phi (eob/seobnrv4phm.py:2319-2372), the likelihood
// all_in_one_likelihood (src/interpolate.cu:553-628) with the host finish in
// get_ll (eob/seobnrv4phm.py:772-823).
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <map>
#include <mutex>
#include <tuple>
#include <utility>

#include "eob_fastmath.hpp"
#include "eobhip_common.hpp"
#include "resample.hpp"
#include "spline_nak.hpp"

using namespace eobhip_detail;

namespace {

constexpr int kBlock = 256;
constexpr double kPi = 3.141592653589793;


// The interior form of a row from its two intervals (spacing, slope); its right-hand
// side without the factor 3.
__device__ __forceinline__ Row interior_row(double d1, double m1, double d2, double m2) {
    Row r;
    r.b = d2 * m1 + d1 * m2;
    r.dg = 2 * (d1 + d2);
    r.ud = d1;
    r.ld = d2;
    return r;
}

// v / d from r = 1 / d: the product and one correction, which rounds as the division
// does for normal numbers (Markstein's method).  With plain products, and 3 times a
// right-hand side rounded before it is used, the coefficients' error against extended
// precision was 4 to 25 % larger (rms; 1.5 to 2 times between the knots of uneven
// chirps) than one elimination from the first row leaves; this way it is equal.  (Halo
// rows keep the products: what they round is damped before it reaches a lane's own.)
__device__ __forceinline__ double over(double v, double d, double r) {
    const double w = v * r;
    return fma(fma(-d, w, v), r, w);
}

// How far from its own rows a lane starts its eliminations (see the batched
// builder below, which explains the bound).
constexpr int kHalo = 32, kHaloMax = 64;
constexpr double kDamped = 0x1p-54;

// Drop-in layout: t [len][nbin], y/B/diagonals [len][ninterp], interpolant
// j = sub * nbin + bin.  A lane takes kDropOwn rows of one interpolant, closed
// between an elimination from below and one from above; lanes run over
// interpolants, so every row is one coalesced access.  grid (interpolants / 64,
// chunks): the lengths are on the device, so a block's wavefronts step through
// the chunks.  Bound by the latency of the eliminated rows (two dependent
// divisions each): 352 series of 2048 knots took 3.65 ms with one lane per
// series, 48 us now.
constexpr int kDropOwn = 32;
struct DropColumn {
    const double *t, *y;
    size_t nbin, ni;
    int len;
    __device__ __forceinline__ double T(int i) const { return t[(size_t)i * nbin]; }
    __device__ __forceinline__ double Y(int i) const { return y[(size_t)i * ni]; }
    __device__ __forceinline__ Row end(int i) const {
        const int j = i == 0 ? 0 : len - 3;
        return nak_row(i, len, T(j), T(j + 1), T(j + 2), Y(j), Y(j + 1), Y(j + 2));
    }
};

__global__ __launch_bounds__(kBlock) void k_interpolate_TD(const double* __restrict__ t, const double* __restrict__ y, double* B,
                                                           double* ud, double* dg, double* ld, const int* __restrict__ lengths,
                                                           int nbin, int ninterp) {
    const int it = blockIdx.x * 64 + (threadIdx.x & 63);
    if (it >= ninterp) return;
    const int b = it % nbin;
    const int len = lengths[b];
    if (len < 3) return;
    const DropColumn c{t + b, y + it, (size_t)nbin, (size_t)ninterp, len};
    const int step = gridDim.y * (kBlock / 64);
    for (int ch = blockIdx.y * (kBlock / 64) + (threadIdx.x >> 6); ch < (len + kDropOwn - 1) / kDropOwn; ch += step) {
        const int s0 = ch * kDropOwn, e0 = s0 + kDropOwn < len ? s0 + kDropOwn : len;
        // rows are eliminated as D s + (the neighbour's coefficient) s' = B, a quotient each
        // from above: Da s_{e0} + la s_{e0-1} = Ba, ia = 1 / Da
        double Da = 1.0, ia = 1.0, Ba = 0.0, la = 0.0;
        for (int halo = kHalo; e0 < len; halo = kHaloMax) {
            const int hi = e0 + halo < len ? e0 + halo : len;
            double damp = hi == len ? 0.0 : 1.0;
            Da = ia = 1.0;
            Ba = la = 0.0;
            double tp = c.T(hi < len ? hi : len - 1), yp = c.Y(hi < len ? hi : len - 1);
            double t0 = c.T(hi - 1), y0 = c.Y(hi - 1);
            double d2 = tp - t0, m2 = (yp - y0) / d2;
#pragma unroll 4
            for (int i = hi - 1; i >= e0; --i) {
                const double tm = c.T(i - 1), ym = c.Y(i - 1);
                const double d1 = t0 - tm, m1 = (y0 - ym) / d1;
                Row r = interior_row(d1, m1, d2, m2);
                double three = 3.0;
                if (i == len - 1) {
                    r = c.end(i);
                    three = 1.0;
                }
                const double w = i == hi - 1 ? 0.0 : r.ud * ia;
                Da = r.dg - w * la;
                Ba = fma(three, r.b, -(w * Ba));   // 3 r.b is not rounded by itself
                la = r.ld;
                ia = 1.0 / Da;
                damp *= r.ud * ia;
                t0 = tm; y0 = ym; d2 = d1; m2 = m1;
            }
            if (fabs(damp) < kDamped || halo == kHaloMax) break;
        }
        // from below: D s_{s0-1} + u s_{s0} = Bb, id = 1 / D
        double D = 1.0, id = 1.0, Bb = 0.0, u = 0.0, t0 = 0.0, y0 = 0.0, d1 = 1.0, m1 = 0.0;
        for (int halo = kHalo;; halo = kHaloMax) {
            const int lo = s0 - halo > 0 ? s0 - halo : 0;
            double damp = lo == 0 ? 0.0 : 1.0;
            D = id = 1.0;
            Bb = u = 0.0;
            t0 = c.T(lo);
            y0 = c.Y(lo);
            if (lo > 0) {
                d1 = t0 - c.T(lo - 1);
                m1 = (y0 - c.Y(lo - 1)) / d1;
            }
#pragma unroll 4
            for (int i = lo; i < s0; ++i) {
                const double tp = c.T(i + 1), yp = c.Y(i + 1);
                const double d2 = tp - t0, m2 = (yp - y0) / d2;
                Row r = interior_row(d1, m1, d2, m2);
                double three = 3.0;
                if (i == 0) {
                    r = c.end(0);
                    three = 1.0;
                }
                const double w = i == lo ? 0.0 : r.ld * id;
                D = r.dg - w * u;
                Bb = fma(three, r.b, -(w * Bb));
                u = r.ud;
                id = 1.0 / D;
                damp *= r.ld * id;
                t0 = tp; y0 = yp; d1 = d2; m1 = m2;
            }
            if (fabs(damp) < kDamped || halo == kHaloMax) break;
        }
        // the lane's rows, then back through them
        double Ds[kDropOwn], Bs[kDropOwn], last_ld = 0.0;
#pragma unroll
        for (int j = 0; j < kDropOwn; ++j) {
            const int i = s0 + j;
            if (i < e0) {
                const int k = i < len - 1 ? i + 1 : i;
                const double tp = c.T(k), yp = c.Y(k);
                const double d2 = tp - t0, m2 = (yp - y0) / d2;
                Row r = interior_row(d1, m1, d2, m2);
                double three = 3.0;
                if (i == 0 || i == len - 1) {
                    r = c.end(i);
                    three = 1.0;
                }
                const double w = over(r.ld, D, id);   // row 0: ld = 0
                D = r.dg - w * u;
                Bb = fma(three, r.b, -(w * Bb));
                u = r.ud;
                id = 1.0 / D;
                last_ld = r.ld;
                t0 = tp; y0 = yp; d1 = d2; m1 = m2;
            }
            Ds[j] = D;
            Bs[j] = Bb;
        }
        const double w = over(u, Da, ia);
        double xi = (Bb - w * Ba) / (D - w * la), xn = (Ba - la * xi) / Da;
        double tn = c.T(e0 < len ? e0 : len - 1), yn = c.Y(e0 < len ? e0 : len - 1), ti = c.T(e0 - 1);
#pragma unroll
        for (int j = kDropOwn - 1; j >= 0; --j) {
            const int i = s0 + j;
            if (i < e0) {
                const double tm = c.T(i > 0 ? i - 1 : 0), yi = c.Y(i);
                if (i < e0 - 1) {
                    const double ui = i > 0 ? ti - tm : c.end(0).ud;
                    xi = over(Bs[j] - ui * xn, Ds[j], 1.0 / Ds[j]);
                }
                const size_t o = (size_t)i * ninterp + it;
                B[o] = xi;
                if (i < len - 1) {
                    const double dt = tn - ti, slope = (yn - yi) / dt;
                    const double tt = (xi + xn - 2 * slope) / dt;
                    ud[o] = xi;
                    dg[o] = (slope - xi) / dt - tt;
                    ld[o] = tt / dt;
                } else {
                    // the last row keeps the eliminated system's values, as the reference leaves them
                    ud[o] = 0.0;
                    dg[o] = D;
                    ld[o] = last_ld;
                }
                xn = xi; tn = ti; yn = yi; ti = tm;
            }
        }
    }
}

// ---------------------------------------------------- batched EOB splines
// nser interpolants per binary over its trajectory knots t_k (units of M):
// knots [n][max_step][nser] (for the (2,2) pipeline nser = 3: phi, Re and Im of
// h22 e^{2 i phi}), coef [n][max_step][4 nser] = (y, c1, c2, c3) per interpolant.
//
// ------------------------------------------------ (2,2) pipeline: tiles
// The three interpolants of the likelihood pipeline's (2,2) mode (and any three
// series on long knots).  The work is split by tiles of kTile rows of one
// binary.  The block forms the tile's spacings and slopes from rows loaded in
// order, once, in LDS; lane c of wavefront q then solves rows 16 c .. 16 c + 15
// of series q: it eliminates the kHalo rows below its own upwards and the kHalo
// rows above downwards, side by side (two independent chains) and both from a
// cut system, closes its own 16 rows between the two and puts their knot slopes
// in LDS, from which the block writes the coefficients in memory order.
//
// The effect of a cut is damped as the sweep kernel's comment below says; the
// lane multiplies the damping factors of its own halo rows, and where their
// product is not below 2^-54 (spacings that shrink over tens of rows) it starts
// again kHaloMax = 64 rows away, where the dominance alone gives 2^-64.  The
// not-a-knot end rows are never cut.
//
// Bound by memory: per knot t (its trajectory row's 40 bytes), the series (8
// bytes each) and the coefficients (32 bytes per series) once each; the halos
// cost five eliminated rows per row but read LDS.  512 chirps of 5k-60k knots
// (16.6 M knots, 160 bytes each): 2.23 ms for the sweep kernel (one wavefront
// per binary, each lane a 21st of the rows, read from memory as it goes),
// 0.60 now; 256 trajectories of 600 knots: 176 and 39 us.
constexpr int kTile = 1024;              // rows per block
constexpr int kOwn = 16;                 // rows per lane
constexpr int kTileSeries = 3;           // one wavefront each
constexpr int kTileThreads = 64 * kTileSeries;
constexpr int kTileRows = kTile + 2 * (kHaloMax + 1);
constexpr int kTileWords = kTileRows + kTileRows / kOwn + 1;   // one word of padding per kOwn rows
static_assert(kTile / kOwn == 64, "one wavefront per series");
__device__ __forceinline__ int tile_at(int k) { return k + (k >> 4); }

// One elimination row: from the neighbour's relation s_n = g - h s (g, h in, cut
// rows g = h = 0) and the row a s_n + dg s + c s_next = k b to s = b' - c' s_next.
struct Carry {
    double h, g;   // c', d'
    // kHalo: a row that is not the lane's own
    template <bool kHalo = true>
    __device__ __forceinline__ double step(double a, double dg, double c, double b, double k = 3.0) {
        const double den = dg - a * h, inv = eob::refined_rcp(den), r = fma(k, b, -(a * g));
        g = kHalo ? r * inv : over(r, den, inv);
        h = kHalo ? c * inv : over(c, den, inv);
        return inv;
    }
};

__global__ __launch_bounds__(kTileThreads) void k_spline_build_tile(const double* __restrict__ dense, const double* __restrict__ knots,
                                                                   const int* __restrict__ num_steps, int max_step,
                                                                   double* __restrict__ coef) {
    constexpr int G = kTileSeries;
    __shared__ double dx[kTileWords], mq[G][kTileWords];
    const int b = blockIdx.y;
    const int len = num_steps[b];
    const int base = blockIdx.x * kTile;
    if (base >= len) return;
    const int tid = threadIdx.x;
    const double* T = dense + (size_t)b * max_step * 5;
    const double* Y = knots + (size_t)b * max_step * G;
    double* C = coef + (size_t)b * max_step * (4 * G);
    if (len < 3) {
        if (tid < G)
            for (int i = 0; i < len; ++i) {
                double* c = C + (size_t)(4 * G) * i + 4 * tid;
                c[0] = Y[(size_t)G * i + tid];
                c[1] = c[2] = c[3] = 0.0;
            }
        return;
    }
    // intervals lo .. top: what the lanes' halos can reach
    const int lo = base - kHaloMax - 1 > 0 ? base - kHaloMax - 1 : 0;
    const int top = base + kTile + kHaloMax < len - 2 ? base + kTile + kHaloMax : len - 2;
    for (int k = tid; k <= top - lo; k += kTileThreads) {
        const double* t = T + (size_t)5 * (lo + k);
        const double* y = Y + (size_t)G * (lo + k);
        const double d = t[5] - t[0];
        dx[tile_at(k)] = d;
#pragma unroll
        for (int q = 0; q < G; ++q) mq[q][tile_at(k)] = eob::qdiv(y[G + q] - y[q], d);
    }
    __syncthreads();
    const int q = tid >> 6, s0 = base + (tid & 63) * kOwn;
    const bool on = s0 < len;
    double x[kOwn + 1];
    if (on) {
        const double* m = mq[q];
        const auto D = [&](int i) { return dx[tile_at(i - lo)]; };
        const auto M = [&](int i) { return m[tile_at(i - lo)]; };
        const int e0 = s0 + kOwn < len ? s0 + kOwn : len;
        Carry dn, up;   // dn: s_{s0-1} = g - h s_{s0}; up: s_{e0} = g - h s_{e0-1}
        // the not-a-knot rows at either end, for the lanes that reach them
        double fb = 0.0, fdg = 1.0, fud = 0.0, lb = 0.0, ldg = 1.0, lld = 0.0;
        if (s0 <= kHaloMax) {
            const double p = D(0), r = D(1), u = M(0), v = M(1), e = p + r;
            fb = ((p + 2 * e) * r * u + p * p * v) / e;
            fud = e;
            fdg = r;
        }
        if (e0 + kHaloMax >= len) {
            const double p = D(len - 3), r = D(len - 2), u = M(len - 3), v = M(len - 2), e = p + r;
            lb = (r * r * u + (2 * e + r) * p * v) / e;
            ldg = p;
            lld = e;
        }
        double d1 = 0.0, m1 = 0.0;   // interval s0 - 1
#pragma unroll 1
        for (int halo = kHalo;; halo = kHaloMax) {
            const int i0 = s0 - halo > 0 ? s0 - halo : 0, i9 = e0 + halo < len ? e0 + halo : len;
            double down = 0.0, above = 0.0;   // damping
            dn.h = dn.g = up.h = up.g = 0.0;
            double a1 = 0.0, am = 0.0, c2 = 0.0, cm = 0.0;
            if (s0 > 0) {
                if (i0 == 0) {
                    a1 = D(0);
                    am = M(0);
                    dn.step(0.0, fdg, fud, fb, 1.0);
                } else {
                    const double b1 = D(i0 - 1), bm = M(i0 - 1);
                    a1 = D(i0);
                    am = M(i0);
                    down = a1 * dn.step(0.0, 2 * (b1 + a1), b1, a1 * bm + b1 * am);
                }
            }
            if (e0 < len) {
                c2 = D(i9 - 2);
                cm = M(i9 - 2);
                if (i9 == len) {
                    up.step(0.0, ldg, lld, lb, 1.0);
                } else {
                    const double b2 = D(i9 - 1), bm = M(i9 - 1);
                    above = c2 * up.step(0.0, 2 * (c2 + b2), b2, b2 * cm + c2 * bm);
                }
            }
            // row i below: intervals i - 1 (a1, am) and i; row j above: j - 1 and j (c2, cm)
#pragma unroll 4
            for (int k = 1; k < halo; ++k) {
                const int i = i0 + k, j = i9 - 1 - k;
                if (i < s0) {
                    const double d2 = D(i), m2 = M(i);
                    down *= d2 * dn.step(d2, 2 * (a1 + d2), a1, d2 * am + a1 * m2);
                    a1 = d2;
                    am = m2;
                }
                if (j >= e0) {
                    const double d0 = D(j - 1), m0 = M(j - 1);
                    above *= d0 * up.step(d0, 2 * (d0 + c2), c2, c2 * m0 + d0 * cm);
                    c2 = d0;
                    cm = m0;
                }
            }
            d1 = a1;
            m1 = am;
            if ((fabs(down) < kDamped && fabs(above) < kDamped) || halo == kHaloMax) break;
        }
        // the lane's rows, then back through them
        double pcs[kOwn], pds[kOwn];
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
            const int i = s0 + j;
            if (i < e0) {
                const int k = i < len - 1 ? i : len - 2;
                const double d2 = D(k), m2 = M(k);
                const bool first = i == 0, last = i == len - 1;
                const double a = first ? 0.0 : (last ? lld : d2), dg = first ? fdg : (last ? ldg : 2 * (d1 + d2));
                const double c = first ? fud : (last ? 0.0 : d1), r = first ? fb : (last ? lb : d2 * m1 + d1 * m2);
                dn.step<false>(a, dg, c, r, first || last ? 1.0 : 3.0);
                d1 = d2;
                m1 = m2;
            }
            pcs[j] = dn.h;   // past the end: the last row's
            pds[j] = dn.g;
        }
        // row e0 - 1: s = g - h s_{e0} with s_{e0} = up.g - up.h s
        double xi = (dn.g - dn.h * up.g) / (1.0 - dn.h * up.h);
        double xn = up.g - up.h * xi;
        x[kOwn] = xn;
#pragma unroll
        for (int j = kOwn - 1; j >= 0; --j) {
            const int i = s0 + j;
            if (i < e0 - 1) xi = pds[j] - pcs[j] * xn;
            x[j] = xi;
            if (i < e0) xn = xi;
        }
    }
    __syncthreads();   // every lane has read the slopes of its halos
    // the knot slopes take the intervals' place: row i at word i - base
    if (on) {
        const int c0 = (tid & 63) * kOwn;
#pragma unroll
        for (int j = 0; j < kOwn; ++j) mq[q][tile_at(c0 + j)] = x[j];
        if ((tid & 63) == 63) mq[q][tile_at(kTile)] = x[kOwn];   // the row past the tile
    }
    __syncthreads();
    const int rows = len - base < kTile ? len - base : kTile;
    const int p = tid % G;
    for (int j = tid / G; j < rows; j += kTileThreads / G) {
        const int i = base + j;
        const double* y = Y + (size_t)G * i + p;
        const double yi = y[0];
        double c1 = 0.0, c2 = 0.0, c3 = 0.0;
        if (i < len - 1) {
            const double xi = mq[p][tile_at(j)], xn = mq[p][tile_at(j + 1)];
            const double dt = dx[tile_at(i - lo)], rt = eob::refined_rcp(dt);
            const double slope = over(y[G] - yi, dt, rt);
            const double tt = over(xi + xn - 2 * slope, dt, rt);
            c1 = xi;
            c2 = over(slope - xi, dt, rt) - tt;
            c3 = over(tt, dt, rt);
        }
        double* c = C + (size_t)(4 * G) * i + 4 * p;
        c[0] = yi;
        c[1] = c1;
        c[2] = c2;
        c[3] = c3;
    }
}

// ------------------------------------------ any number of series: sweeps
// The higher modes' series and those of r and pr.  These feed the
// merger-ringdown attachment, whose discrete choices (the knot of the
// frequency's peak, the attachment sample) turn on the last bits of the
// coefficients for some binaries, so their order of operations is kept.
//
// One wavefront per binary builds all of them.  Each interpolant's slope
// system is split into P <= 64 / nser chunks of >= kChunkMin rows, one lane
// per (interpolant, chunk); the lane solves its chunk together with kHalo rows on either side as
// a system of its own (cut off where the halo ends) and keeps the slopes of its
// own rows.  Inside the system every row is diagonally dominant (2(dx1 + dx2)
// against dx1 + dx2), so the effect of the cut on a row k rows away is damped
// by at least 2^-k, and by 0.268^k on evenly spaced knots: with 32 halo rows
// it is below 5e-19 of the neighbouring slopes on even knots and 2e-10 in the
// worst case the dominance allows (every spacing shrinking by a large factor
// over 32 rows, which an adaptive step sequence cannot do).  Emulated on the
// CPU against the uncut solve, 32 halo rows give the same coefficients as 64
// to rounding on trajectory knots (spacing ratio 33 where the fixed-step pass
// begins) and on 5k-60k-knot chirps; 24 rows already move them by 1e-14.  The
// not-a-knot end rows are never cut.
//
// Nothing of the system goes to memory: the rows are formed from t and y as the
// sweeps reach them, the forward elimination keeps only its carry (c', d') at
// the start of every kSeg rows (a checkpoint, 16 bytes per kSeg rows), and the
// back substitution walks the segments top down, recomputing each segment's
// (c', d') in registers from its checkpoint and writing the polynomial
// coefficients of each interval as soon as both end slopes are known.  Memory
// traffic is t and y read once and the coefficients written once (the
// recomputation and the halos re-read rows from the caches).
constexpr int kChunkMin = 96;
constexpr int kSplineLanes = 64;
constexpr int kSeg = 16;
constexpr int kMaxSeries = 32;

__host__ __device__ inline int spline_chunks(int len, int nser) {
    const int pmax = kSplineLanes / nser;
    int P = len / kChunkMin;
    return P < 1 ? 1 : (P > pmax ? pmax : P);
}
// checkpoints per lane for a binary of len knots (segments of its chunk's sweep)
__host__ __device__ inline int spline_segs(int len, int nser) {
    const int P = spline_chunks(len, nser);
    const int m = (len + P - 1) / P;
    return (m + 2 * kHalo + kSeg - 1) / kSeg + 1;
}
// doubles per binary: nser P lanes x 2 doubles x spline_segs for every len <=
// max_step (nser P 2 segs <= 2 nser len / kSeg + 2 P nser (1 + 2 kHalo) / kSeg +
// 4 P nser with P nser <= 64; checked for nser <= 32 and every len up to 70000)
__host__ __device__ inline long long spline_scratch_per_bin(int max_step, int nser) {
    return (2LL * nser * max_step + 2LL * kSplineLanes * (2 * kHalo + 2 * kSeg)) / kSeg + 4 * kSplineLanes + 64;
}

// t and y of rows start-2 .. start+kSeg+1, clamped into [0, len-1]; issued together
__device__ __forceinline__ void seg_load(const double* __restrict__ T, const double* __restrict__ Y, int ys, int start, int len,
                                         double* wt, double* wy) {
#pragma unroll
    for (int k = 0; k < kSeg + 4; ++k) {
        int i = start - 2 + k;
        i = i < 0 ? 0 : (i > len - 1 ? len - 1 : i);
        wt[k] = T[5 * i];
        wy[k] = Y[(size_t)ys * i];
    }
}

// Forward elimination over rows start .. end-1 (end - start <= kSeg) of the
// system cut to rows lo .. hi-1, from the carry (pc, pd) of the row below;
// kKeep stores every row's (c', d').  Interior row i = start + j reads the
// window at j+1, j+2, j+3 (rows i-1, i, i+1); the two end rows (rfirst, rlast)
// are formed once by the caller and picked by value, so that every window
// index stays a compile-time constant (a select between window entries would
// turn into a computed address and push the window out of registers).
template <bool kKeep>
__device__ __forceinline__ void seg_forward(const double* wt, const double* wy, int start, int end, int lo, int hi, int len,
                                            const Row& rfirst, const Row& rlast, double& pc, double& pd, double* pcs, double* pds) {
#pragma unroll
    for (int j = 0; j < kSeg; ++j) {
        const int i = start + j;
        if (i < end) {
            Row r = nak_row(1, 3, wt[j + 1], wt[j + 2], wt[j + 3], wy[j + 1], wy[j + 2], wy[j + 3]);   // the interior form
            if (i == 0) r = rfirst;
            if (i == len - 1) r = rlast;
            const double a = (i == lo) ? 0.0 : r.ld;        // cut below the halo
            const double c = (i == hi - 1) ? 0.0 : r.ud;    // cut above the halo
            const double den = r.dg - a * pc;
            pc = c / den;
            pd = (r.b - a * pd) / den;
            if constexpr (kKeep) {
                pcs[j] = pc;
                pds[j] = pd;
            }
        }
    }
}

__global__ __launch_bounds__(kSplineLanes) void k_spline_build_seg(const double* __restrict__ dense, const double* __restrict__ knots,
                                                                   const int* __restrict__ num_steps, int n, int max_step, int nser,
                                                                   double* __restrict__ coef, double* __restrict__ scratch) {
    const int b = blockIdx.x;
    if (b >= n) return;
    const int len = num_steps[b];
    const int lane = threadIdx.x;
    const int cs = 4 * nser;   // coefficient row stride
    const double* T = dense + (size_t)b * max_step * 5;
    if (len < 3) {
        if (lane < nser) {
            const double* Y = knots + (size_t)b * max_step * nser + lane;
            double* C = coef + (size_t)b * max_step * cs + 4 * lane;
            for (int i = 0; i < len; ++i) {
                C[(size_t)cs * i] = Y[(size_t)nser * i];
                C[(size_t)cs * i + 1] = C[(size_t)cs * i + 2] = C[(size_t)cs * i + 3] = 0.0;
            }
        }
        return;
    }
    const int P = spline_chunks(len, nser);
    if (lane >= nser * P) return;
    const int q = lane / P, cidx = lane % P;
    const double* Y = knots + (size_t)b * max_step * nser + q;
    double* C = coef + (size_t)b * max_step * cs + 4 * q;
    const int m = (len + P - 1) / P;
    const int s0 = cidx * m, e0 = (s0 + m < len) ? s0 + m : len;
    if (s0 >= e0) return;
    const int lo = (s0 - kHalo > 0) ? s0 - kHalo : 0;
    const int hi = (e0 + kHalo < len) ? e0 + kHalo : len;
    const int nseg = (hi - lo + kSeg - 1) / kSeg;
    double* ck = scratch + (size_t)b * spline_scratch_per_bin(max_step, nser) + (size_t)lane * 2 * spline_segs(len, nser);
    const Row rfirst = nak_row(0, len, T[0], T[5], T[10], Y[0], Y[nser], Y[2 * nser]);
    const Row rlast = nak_row(len - 1, len, T[5 * (len - 3)], T[5 * (len - 2)], T[5 * (len - 1)], Y[(size_t)nser * (len - 3)],
                              Y[(size_t)nser * (len - 2)], Y[(size_t)nser * (len - 1)]);
    // the next segment's rows (and checkpoint) are loaded while this one is
    // eliminated: the sweeps are chains of dependent divisions, and without the
    // prefetch each segment would wait a memory round trip for its rows
    double wt[kSeg + 4], wy[kSeg + 4], nt[kSeg + 4], ny[kSeg + 4];
    double pc = 0.0, pd = 0.0;
    seg_load(T, Y, nser, lo, len, wt, wy);
    for (int sg = 0; sg < nseg; ++sg) {
        const int start = lo + sg * kSeg, end = (start + kSeg < hi) ? start + kSeg : hi;
        ck[2 * sg] = pc;
        ck[2 * sg + 1] = pd;
        if (sg + 1 < nseg) seg_load(T, Y, nser, start + kSeg, len, nt, ny);
        seg_forward<false>(wt, wy, start, end, lo, hi, len, rfirst, rlast, pc, pd, nullptr, nullptr);
        if (sg + 1 < nseg) {
#pragma unroll
            for (int k = 0; k < kSeg + 4; ++k) { wt[k] = nt[k]; wy[k] = ny[k]; }
        }
    }
    // back substitution, segment by segment from the top; xn = slope of the row above
    double xn = 0.0;
    int sg = nseg - 1;
    seg_load(T, Y, nser, lo + sg * kSeg, len, wt, wy);
    double cpc = ck[2 * sg], cpd = ck[2 * sg + 1];
    for (; sg >= 0; --sg) {
        const int start = lo + sg * kSeg, end = (start + kSeg < hi) ? start + kSeg : hi;
        if (end <= s0) break;   // the rows below this lane's chunk need no slopes
        double pcs[kSeg], pds[kSeg];
        pc = cpc;
        pd = cpd;
        const bool more = sg > 0 && start > s0;
        if (more) {
            seg_load(T, Y, nser, start - kSeg, len, nt, ny);
            cpc = ck[2 * (sg - 1)];
            cpd = ck[2 * (sg - 1) + 1];
        }
        seg_forward<true>(wt, wy, start, end, lo, hi, len, rfirst, rlast, pc, pd, pcs, pds);
#pragma unroll
        for (int j = kSeg - 1; j >= 0; --j) {
            const int i = start + j;
            if (i < end) {
                const double xi = pds[j] - pcs[j] * xn;   // the cut row hi-1 has c' = 0
                if (i >= s0 && i < e0) {
                    double* c = C + (size_t)cs * i;
                    if (i < len - 1) {
                        const double yi = wy[j + 2], yp = wy[j + 3];
                        const double dt = wt[j + 3] - wt[j + 2];
                        const double slope = (yp - yi) / dt;
                        const double tt = (xi + xn - 2 * slope) / dt;
                        c[0] = yi;
                        c[1] = xi;
                        c[2] = (slope - xi) / dt - tt;
                        c[3] = tt / dt;
                    } else {
                        c[0] = wy[j + 2];
                        c[1] = c[2] = c[3] = 0.0;
                    }
                }
                xn = xi;
            }
        }
        if (!more) break;
#pragma unroll
        for (int k = 0; k < kSeg + 4; ++k) { wt[k] = nt[k]; wy[k] = ny[k]; }
    }
}

// Uniform resample of h+ = amp * Re[(Re S + i Im S)(t) e^{-2 i phi(t)}] at
// t_j = t_0 + j dT_M (dT_M = dt / (M MTSUN)), j < N_b = floor((t_last - t_0)/dT_M) + 1,
// zero for N_b <= j < N; hx is the imaginary part, the two series the reference
// transforms (eob/seobnrv4phm.py:720, 742-744).  grid (blocks, binaries), a run
// of samples per wavefront (resample.hpp).  Bound by the writes: 256 binaries x
// 2^20 samples, 10% of them inside a template: h+ 593 us with knot windows per
// block, 412 interval by interval, 373 now (a fill of the same memory 340).
// samples with a value: floor((t_last - t_0) / dT) + 1, at most N
__device__ __forceinline__ long long series_samples(const double* T, int len, double dT, int N) {
    if (len < 2) return 0;
    const long long nb = (long long)((T[5 * (len - 1)] - T[0]) / dT) + 1;
    return nb > N ? N : nb;
}

constexpr int kH22Room = 12 * kMostStaged;   // doubles a wavefront stages
template <int kRows>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_resample_hplus(const double* __restrict__ dense, const double* __restrict__ coef,
                                                           const int* __restrict__ num_steps, const double* __restrict__ amp,
                                                           const double* __restrict__ dT_M, int max_step, int N,
                                                           double* __restrict__ hplus, int* __restrict__ nsamp,
                                                           double* __restrict__ hcross) {
    const int b = blockIdx.y;
    const int len = num_steps[b];
    const double* T = dense + (size_t)b * max_step * 5;
    const double dT = dT_M[b];
    const long long nb = series_samples(T, len, dT, N);
    if (blockIdx.x == 0 && threadIdx.x == 0) nsamp[b] = (int)nb;
    const SeriesOut<> o{hplus + (size_t)b * N, hcross ? hcross + (size_t)b * N : nullptr, amp[b], nb, N};
    const double* C = coef + (size_t)b * max_step * 12;
    const double t0 = T[0];
    extern __shared__ __attribute__((aligned(16))) double staged[];
    double* st = staged + wave_index() * kH22Room;
    for_runs(N, kRows, blockIdx.x, gridDim.x, [&](long long j0) {
        if (j0 < nb)
            h22_rows(st, kRows, kMostStaged, true, T, C, len, t0, dT, j0, nb,
                     [&](long long j, const double (&re)[2], const double (&im)[2], bool full) { o.put(j, re, im, full); });
        o.zeros(j0, kRows);
    });
}

// Uniform resample of the mode sum h = amp sum_j S_j(t) e^{-i m_j phi(t)} (the
// reference's modes *= exp(-1j m phi_interp) and template = modes.sum,
// eob/seobnrv4phm.py:2366-2372, 720) at t_j = t_0 + j dT_M, j < N_b, zero past;
// hplus, hcross = Re h, Im h (the two series it transforms, :742-744).  coef
// [n][max_step][4 (2 nm + 1)]: series j < nm Re S_j, nm + j Im S_j, 2 nm phi.
// e^{-i m phi} is formed as the m-th power of e^{-i phi}.
constexpr int kMaxModeM = 8;
// One sample's sum from a row (Re of each mode, Im of each mode, phi; 4
// coefficients per series), by Horner's rule in e^{-i phi} over the modes by
// falling m: a mode costs the products between its m and the next one's.
template <Phases P, class Ptr>
__device__ __forceinline__ bool modes_sample(Ptr c, double x, int nm, const ModeOrder& mo, double& hr, double& hi) {
    const double x2 = x * x, x3 = x2 * x;
    const auto cubic = [&](Ptr p) { return p[0] + p[1] * x + p[2] * x2 + p[3] * x3; };
    double sp, cph;
    const bool good = sincos_of<P>(cubic(c + 4 * (2 * nm)), sp, cph);
    double r = 0.0, i = 0.0;
    const auto turn = [&](int k) {
        for (; k > 0; --k) {
            const double t = r * cph + i * sp;
            i = i * cph - r * sp;
            r = t;
        }
    };
#pragma unroll 1
    for (int k = 0; k < nm; ++k) {
        const int q = mo.q(k);
        turn(mo.down(k));
        r += cubic(c + 4 * q);
        i += cubic(c + 4 * (nm + q));
    }
    turn(mo.down(nm));
    hr = r;
    hi = i;
    return good;
}

// Five modes of 512 binaries x 2^20, 10% of the samples inside a template: 2470 us with
// knot windows per block, 1520 interval by interval, 1470 to 1570 now (the writes alone
// 1360).  One build for any number of modes: what a wavefront stages is 63 rows of one
// mode, 28 of five, 10 of fifteen.
constexpr int kModesRoom = 1264;   // doubles a wavefront stages: four blocks fill a CU's LDS
template <int kRows>
__global__ __launch_bounds__(kBlock) void k_resample_modes(const double* __restrict__ dense, const double* __restrict__ coef,
                                                           const int* __restrict__ num_steps, const double* __restrict__ amp,
                                                           const double* __restrict__ dT_M, int max_step, int N, int nm, ModeOrder mo,
                                                           double* __restrict__ hplus, double* __restrict__ hcross,
                                                           int* __restrict__ nsamp) {
    const int b = blockIdx.y;
    const int len = num_steps[b];
    const int cs = 4 * (2 * nm + 1);
    const double* T = dense + (size_t)b * max_step * 5;
    const double* C = coef + (size_t)b * max_step * cs;
    const double dT = dT_M[b], t0 = T[0];
    const long long nb = series_samples(T, len, dT, N);
    if (blockIdx.x == 0 && threadIdx.x == 0) nsamp[b] = (int)nb;
    const SeriesOut<> o{hplus + (size_t)b * N, hcross + (size_t)b * N, amp[b], nb, N};
    extern __shared__ __attribute__((aligned(16))) double staged[];
    double* st = staged + wave_index() * kModesRoom;
    for_runs(N, kRows, blockIdx.x, gridDim.x, [&](long long j0) {
        if (j0 < nb)
            resample_rows(
                kRows, staged_rows(kModesRoom, cs), true, T, len, j0, nb, [&](long long j) { return t0 + (double)j * dT; },
                [&](int i, int n) { stage_rows<6>(st, C + (size_t)cs * i, n, cs); },
                [&](int k, double x, double& re, double& im) { return modes_sample<kBounded>(st + k * cs, x, nm, mo, re, im); },
                [&](int i, double x, double& re, double& im) { return modes_sample<kBounded>(C + (size_t)cs * i, x, nm, mo, re, im); },
                [&](int i, double x, double& re, double& im) { return modes_sample<kAny>(C + (size_t)cs * i, x, nm, mo, re, im); },
                [&](long long j, const double (&re)[2], const double (&im)[2], bool full) { o.put(j, re, im, full); });
        o.zeros(j0, kRows);
    });
}

// TD2 (src/interpolate.cu:441-549), TDInterp_wrap2's kernel: per binary b and
// sample i < lengths[b], sum over modes of (re + i im) e^{-i m phi} with every
// series evaluated at the caller's interval inds[b][i] (t - ts[b][ind], data
// time dataTime[i] shared by the binaries).  Series s of binary b starts at
// b (2M + 1) old_length + s * stride: stride old_lengths[b] as the reference
// indexes (correct only when every binary fills old_length), or old_length for
// the padded layout (legacy_stride 0).  Intervals are clamped into
// [0, old_length - 1].  grid (blocks over samples, binaries).
__global__ __launch_bounds__(kBlock) void k_td_interp2(double2* __restrict__ out, const double* __restrict__ dataTime,
                                                       const double* __restrict__ ts, const double* __restrict__ y,
                                                       const double* __restrict__ c1, const double* __restrict__ c2,
                                                       const double* __restrict__ c3, int old_length, const int* __restrict__ old_lengths,
                                                       int data_length, int numModes, const int* __restrict__ ms,
                                                       const int* __restrict__ inds, const int* __restrict__ lengths, int max_length,
                                                       int legacy_stride) {
    const int b = blockIdx.y;
    // sample counts and strides are clamped to the arrays' extents (the reference
    // trusts them; for valid inputs the clamps change nothing)
    int n = lengths[b];
    n = n < max_length ? n : max_length;
    n = n < data_length ? n : data_length;
    int olh = old_lengths[b];
    olh = olh < 0 ? 0 : (olh > old_length ? old_length : olh);
    const long long stride = legacy_stride ? olh : old_length;
    const size_t base = (size_t)b * (2 * numModes + 1) * old_length;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        int ind = inds[(size_t)max_length * b + i];
        ind = ind < 0 ? 0 : (ind > old_length - 1 ? old_length - 1 : ind);
        const double x = dataTime[i] - ts[(size_t)b * old_length + ind];
        const double x2 = x * x, x3 = x * x2;
        size_t k = base + (size_t)(2 * numModes) * stride + ind;
        const double phi = y[k] + c1[k] * x + c2[k] * x2 + c3[k] * x3;
        double hr = 0.0, hi = 0.0;
        for (int q = 0; q < numModes; ++q) {
            k = base + (size_t)q * stride + ind;
            const double re = y[k] + c1[k] * x + c2[k] * x2 + c3[k] * x3;
            k = base + (size_t)(numModes + q) * stride + ind;
            const double im = y[k] + c1[k] * x + c2[k] * x2 + c3[k] * x3;
            double s, c;
            sincos(-((double)ms[q] * phi), &s, &c);
            hr += re * c - im * s;
            hi += re * s + im * c;
        }
        out[(size_t)b * data_length + i] = make_double2(hr, hi);
    }
}

// log L_b = -1/2 * 4 df * sum_k |d_k - h_k|^2 / S(f_k), S(f) = (f/f0)^-4 + 1 + (f/f0)^2,
// 1/S(0) = 0.  Stage 1: per (chunk, binary) partial sums with wave shuffles + LDS;
// chunks of one binary are adjacent in blockIdx.x so the data spectrum is read
// once from HBM and reused from L2 by every binary.
constexpr int kLikeBlock = 256;
constexpr int kLikePerThread = 8;
__global__ __launch_bounds__(kLikeBlock) void k_fd_likelihood_partial(const double2* __restrict__ ht, const double2* __restrict__ dt,
                                                                      int n, int F, double df, double f0, double* __restrict__ partial,
                                                                      int nchunks) {
    const int b = blockIdx.x % n;
    const int chunk = blockIdx.x / n;
    const int base = chunk * kLikeBlock * kLikePerThread;
    const double2* h = ht + (size_t)b * F;
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < kLikePerThread; ++u) {
        const int k = base + u * kLikeBlock + threadIdx.x;
        if (k < F) {
            const double2 hv = h[k];
            const double2 dv = dt[k];
            const double re = dv.x - hv.x, im = dv.y - hv.y;
            const double x = df * (double)k / f0;
            const double x2 = x * x, x4 = x2 * x2;
            const double w = (k == 0) ? 0.0 : x4 / (1.0 + x4 + x4 * x2);   // 1 / S(f)
            acc += (re * re + im * im) * w;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    __shared__ double red[kLikeBlock / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kLikeBlock / 64; ++w) s += red[w];
        partial[(size_t)b * nchunks + chunk] = s;
    }
}

__global__ __launch_bounds__(64) void k_fd_likelihood_final(const double* __restrict__ partial, int n, int nchunks, double df,
                                                            double* __restrict__ logl) {
    const int b = blockIdx.x;
    if (b >= n) return;
    double acc = 0.0;
    for (int c = threadIdx.x; c < nchunks; c += 64) acc += partial[(size_t)b * nchunks + c];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (threadIdx.x == 0) logl[b] = -0.5 * 4.0 * df * acc;
}

// Drop-in all_in_one_likelihood: per 1024-bin block partial sums of
// |d - (F+ hp + Fx hc) e^{-2 pi i f dt}|^2 / psd.  One 256-thread block covers
// 1024 bins (4 per thread); grid (bins / 1024, nbin, nchan).
__global__ __launch_bounds__(kBlock) void k_all_in_one_likelihood(double2* temp_sum, const double2* __restrict__ hp,
                                                                  const double2* __restrict__ hc, const double2* __restrict__ data,
                                                                  const double* __restrict__ psd, const double* __restrict__ Fp,
                                                                  const double* __restrict__ Fc, const double* __restrict__ ts,
                                                                  double df, int nbin, int nchan, int F) {
    const int blk = blockIdx.x, b = blockIdx.y, c = blockIdx.z;
    const double fp = Fp[c * nbin + b], fc = Fc[c * nbin + b], tsh = ts[c * nbin + b];
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int k = blk * 1024 + u * kBlock + threadIdx.x;
        if (k < F) {
            const double2 a = hp[(size_t)b * F + k], e = hc[(size_t)b * F + k], d = data[(size_t)c * F + k];
            const double hr = fp * a.x + fc * e.x, hi = fp * a.y + fc * e.y;
            double s, co;
            sincos(-2.0 * kPi * (df * k) * tsh, &s, &co);
            const double rr = d.x - (hr * co - hi * s), ri = d.y - (hr * s + hi * co);
            acc += (rr * rr + ri * ri) / psd[(size_t)c * F + k];
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    __shared__ double red[kBlock / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kBlock / 64; ++w) s += red[w];
        temp_sum[((size_t)blk * nbin + b) * nchan + c] = make_double2(s, 0.0);
    }
}

}  // namespace

namespace eobhip_detail {

// hipFFT plans, cached per (N, rows per call, stream, direction).  A plan owns a
// work area, so two streams never share one: work queued on different streams
// may overlap.  Callers pass rows in chunks of kFftChunk and the rest in
// power-of-two chunks, which bounds the plans per stream and size to seven.
namespace {
std::mutex g_plan_mu;
std::map<std::tuple<long long, int, void*, int>, hipfftHandle> g_plans;
}  // namespace

int fft_exec(int inverse, const void* in, void* out, int rows, int N, void* stream) {
    std::lock_guard<std::mutex> g(g_plan_mu);
    hipfftHandle plan;
    const auto key = std::make_tuple((long long)N, rows, stream, inverse);
    auto itp = g_plans.find(key);
    if (itp == g_plans.end()) {
        int dims[1] = {N};
        hipfftResult r = inverse ? hipfftPlanMany(&plan, 1, dims, nullptr, 1, N / 2 + 1, nullptr, 1, N, HIPFFT_Z2D, rows)
                                 : hipfftPlanMany(&plan, 1, dims, nullptr, 1, N, nullptr, 1, N / 2 + 1, HIPFFT_D2Z, rows);
        if (r != HIPFFT_SUCCESS) {
            set_error("hipfftPlanMany failed (%d)", (int)r);
            return EOBHIP_EHIP;
        }
        r = hipfftSetStream(plan, as_stream(stream));
        if (r != HIPFFT_SUCCESS) {
            set_error("hipfftSetStream failed (%d)", (int)r);
            return EOBHIP_EHIP;
        }
        g_plans[key] = plan;
    } else {
        plan = itp->second;
    }
    hipfftResult r = inverse ? hipfftExecZ2D(plan, reinterpret_cast<hipfftDoubleComplex*>(const_cast<void*>(in)),
                                             static_cast<double*>(out))
                             : hipfftExecD2Z(plan, static_cast<double*>(const_cast<void*>(in)),
                                             reinterpret_cast<hipfftDoubleComplex*>(out));
    if (r != HIPFFT_SUCCESS) {
        set_error("hipfftExec failed (%d)", (int)r);
        return EOBHIP_EHIP;
    }
    return EOBHIP_OK;
}

int fft_rows(int inverse, const void* in, void* out, int n, int N, void* stream) {
    const size_t F = (size_t)N / 2 + 1;
    const size_t in_stride = inverse ? 2 * F : (size_t)N;     // doubles per input row
    const size_t out_stride = inverse ? (size_t)N : 2 * F;    // doubles per output row
    const double* src = static_cast<const double*>(in);
    double* dst = static_cast<double*>(out);
    // the library's own kernels where they apply: lengths 2^10 (the smallest any
    // path here transforms) to 2^21 (A and B of a row up to 2^10).  They are
    // faster at every length there (2^10: 20 us against 370 for 4096 rows, 2^15:
    // 217 against 462 for 1024, 2^21: 1.87 ms against 4.70 for 128; one row of
    // 2^20: 18 us against 44; only up to 64 rows of 2^10 take 5.6 to 6.0 us against
    // 5.3 to 5.7) and need no plan or work area.
    if (!inverse) {
        const int L = rfft_own_log2(in, out, n, N);
        if (L) return rfft_own(src, dst, n, L, as_stream(stream));
    }
    // full chunks of kFftChunk rows, then the rest by its binary digits (32, 16, ..., 1)
    int row = 0;
    for (int chunk = kFftChunk; chunk >= 1; chunk >>= 1) {
        while (row + chunk <= n) {
            const int rc = fft_exec(inverse, src + row * in_stride, dst + row * out_stride, chunk, N, stream);
            if (rc) return rc;
            row += chunk;
            if (chunk < kFftChunk) break;
        }
    }
    return EOBHIP_OK;
}

}  // namespace eobhip_detail

extern "C" {

int eobhip_interpolate_TD(const double* t_arr, const double* propArrays, double* B, double* upper_diag, double* diag, double* lower_diag,
                          const int* lengths, int numBinAll, int nsubs, void* stream) {
    EOBHIP_REQUIRE(numBinAll >= 0 && nsubs >= 0, "bad sizes");
    const int ni = numBinAll * nsubs;
    if (ni == 0) return EOBHIP_OK;
    // chunks in flight per 64 interpolants: about 8192 wavefronts in all
    const unsigned gx = blocks_for(ni, 64), gy = gx < 2048 ? 2048 / gx : 1;
    hipLaunchKernelGGL(k_interpolate_TD, dim3(gx, gy), dim3(kBlock), 0, as_stream(stream), t_arr, propArrays, B, upper_diag, diag,
                       lower_diag, lengths, numBinAll, ni);
    return check_launch("interpolate_TD");
}

int eobhip_all_in_one_likelihood(double* temp_sum, const double* hp_fd, const double* hc_fd, const double* data, const double* psd,
                                 const double* Fplus, const double* Fcross, const double* time_shift, double df, int num_bin_all,
                                 int nchannels, int data_length, void* stream) {
    EOBHIP_REQUIRE(num_bin_all >= 0 && nchannels >= 0 && data_length >= 0, "bad sizes");
    EOBHIP_REQUIRE(num_bin_all <= 65535 && nchannels <= 65535, "num_bin_all and nchannels must be <= 65535");
    if (num_bin_all == 0 || nchannels == 0 || data_length == 0) return EOBHIP_OK;
    const int nblk = (data_length + 1023) / 1024;
    hipLaunchKernelGGL(k_all_in_one_likelihood, dim3(nblk, num_bin_all, nchannels), dim3(kBlock), 0, as_stream(stream),
                       reinterpret_cast<double2*>(temp_sum), reinterpret_cast<const double2*>(hp_fd),
                       reinterpret_cast<const double2*>(hc_fd), reinterpret_cast<const double2*>(data), psd, Fplus, Fcross, time_shift,
                       df, num_bin_all, nchannels, data_length);
    return check_launch("all_in_one_likelihood");
}

size_t eobhip_spline_scratch_doubles(int n, int max_step) {
    if (n < 0 || max_step < 1) return 0;
    return (size_t)n * (size_t)spline_scratch_per_bin(max_step, 3);
}

int eobhip_spline_build_batched(const double* dense, const double* knots, const int* num_steps, int n, int max_step, double* coef,
                                double* scratch, void* stream) {
    (void)scratch;   // the tiles need none
    EOBHIP_REQUIRE(n >= 0 && max_step >= 1, "bad sizes");
    for (int b = 0; b < n; b += 65535) {   // the grid's second dimension
        const int nb = n - b < 65535 ? n - b : 65535;
        hipLaunchKernelGGL(k_spline_build_tile, dim3(blocks_for(max_step, kTile), nb), dim3(kTileThreads), 0, as_stream(stream),
                           dense + (size_t)b * max_step * 5, knots + (size_t)b * max_step * 3, num_steps + b, max_step,
                           coef + (size_t)b * max_step * 12);
        const int rc = check_launch("spline_build");
        if (rc) return rc;
    }
    return EOBHIP_OK;
}

size_t eobhip_spline_series_scratch_doubles(int n, int max_step, int nser) {
    if (n < 0 || max_step < 1 || nser < 1 || nser > kMaxSeries) return 0;
    return (size_t)n * (size_t)spline_scratch_per_bin(max_step, nser);
}

int eobhip_spline_build_series(const double* dense, const double* knots, const int* num_steps, int n, int max_step, int nser,
                               double* coef, double* scratch, void* stream) {
    EOBHIP_REQUIRE(n >= 0 && max_step >= 1, "bad sizes");
    EOBHIP_REQUIRE(nser >= 1 && nser <= kMaxSeries, "nser must be 1 .. 32");
    if (n == 0) return EOBHIP_OK;
    hipLaunchKernelGGL(k_spline_build_seg, dim3(n), dim3(kSplineLanes), 0, as_stream(stream), dense, knots, num_steps, n, max_step, nser,
                       coef, scratch);
    return check_launch("spline_build");
}

int eobhip_resample_hplus(const double* dense, const double* coef, const int* num_steps, const double* amp, const double* dT_M, int n,
                          int max_step, int N, double* hplus, int* nsamp, void* stream) {
    EOBHIP_REQUIRE(n >= 0 && N >= 1 && n <= 65535, "bad sizes");
    if (n == 0) return EOBHIP_OK;
    const ResampleShape s = resample_shape(N, n, kH22Room);
    hipLaunchKernelGGL(s.rows == 1 ? k_resample_hplus<1> : k_resample_hplus<kRunRows>, s.grid, s.block, s.lds, as_stream(stream), dense, coef,
                       num_steps, amp, dT_M, max_step, N, hplus, nsamp, nullptr);
    return check_launch("resample_hplus");
}

int eobhip_resample_modes(const double* dense, const double* coef, const int* num_steps, const double* amp, const double* dT_M, int n,
                          int max_step, int N, int nm, const int* ms, double* hplus, double* hcross, int* nsamp, void* stream) {
    EOBHIP_REQUIRE(n >= 0 && N >= 1 && n <= 65535, "bad sizes");
    EOBHIP_REQUIRE(nm >= 1 && nm <= 15, "nm must be 1 .. 15");
    EOBHIP_REQUIRE(hplus && hcross, "hplus and hcross are required");
    for (int q = 0; q < nm; ++q) EOBHIP_REQUIRE(ms[q] >= 1 && ms[q] <= kMaxModeM, "m must be 1 .. 8");
    if (n == 0) return EOBHIP_OK;
    const ResampleShape s = resample_shape(N, n, kModesRoom);
    hipLaunchKernelGGL(s.rows == 1 ? k_resample_modes<1> : k_resample_modes<kRunRows>, s.grid, s.block, s.lds, as_stream(stream), dense, coef,
                       num_steps, amp, dT_M, max_step, N, nm, mode_order(ms, nm), hplus, hcross, nsamp);
    return check_launch("resample_modes");
}

int eobhip_TDInterp2(void* templateChannels, const double* dataTime, const double* ts, const double* propArrays, const double* c1,
                     const double* c2, const double* c3, int old_length, const int* old_lengths, int data_length, int numBinAll,
                     int numModes, const int* ls, const int* ms, const int* inds, const int* lengths, int max_length, int legacy_stride,
                     void* stream) {
    (void)ls;   // the reference reads ls into shared memory but combines with m only
    EOBHIP_REQUIRE(numBinAll >= 0 && numModes >= 1 && old_length >= 1 && max_length >= 0 && data_length >= 0, "bad sizes");
    EOBHIP_REQUIRE(numBinAll <= 65535, "numBinAll must be <= 65535 (grid y dimension)");
    if (numBinAll == 0 || max_length == 0) return EOBHIP_OK;
    int bx = (max_length + kBlock - 1) / kBlock;
    if (bx > 4096) bx = 4096;
    hipLaunchKernelGGL(k_td_interp2, dim3(bx, numBinAll), dim3(kBlock), 0, as_stream(stream), static_cast<double2*>(templateChannels),
                       dataTime, ts, propArrays, c1, c2, c3, old_length, old_lengths, data_length, numModes, ms, inds, lengths, max_length,
                       legacy_stride);
    return check_launch("TDInterp2");
}

int eobhip_resample_hpc(const double* dense, const double* coef, const int* num_steps, const double* amp, const double* dT_M, int n,
                        int max_step, int N, double* hplus, double* hcross, int* nsamp, void* stream) {
    EOBHIP_REQUIRE(n >= 0 && N >= 1 && n <= 65535, "bad sizes");
    EOBHIP_REQUIRE(hcross != nullptr, "hcross is required");
    if (n == 0) return EOBHIP_OK;
    const ResampleShape s = resample_shape(N, n, kH22Room);
    hipLaunchKernelGGL(s.rows == 1 ? k_resample_hplus<1> : k_resample_hplus<kRunRows>, s.grid, s.block, s.lds, as_stream(stream), dense, coef,
                       num_steps, amp, dT_M, max_step, N, hplus, nsamp, hcross);
    return check_launch("resample_hpc");
}

// Batched real-to-complex FFT of n rows of N samples into n rows of N/2+1 bins (no dt factor,
// as the reference's rfft, eob/seobnrv4phm.py:742-744).
int eobhip_rfft_batched(const double* in, double* out, int n, int N, void* stream) {
    EOBHIP_REQUIRE(n >= 1 && N >= 2 && (N % 2) == 0, "bad sizes (n >= 1, N even)");
    return fft_rows(0, in, out, n, N, stream);
}

int eobhip_fd_likelihood(const double* htilde, const double* dtilde, double* partial, int n, int F, double df, double f0,
                         double* logl, void* stream) {
    EOBHIP_REQUIRE(n >= 1 && F >= 1, "bad sizes");
    const int per = kLikeBlock * kLikePerThread;
    const int nchunks = (F + per - 1) / per;
    const long long grid = (long long)nchunks * n;
    EOBHIP_REQUIRE(grid < (1LL << 31), "grid too large");
    hipLaunchKernelGGL(k_fd_likelihood_partial, dim3((unsigned)grid), dim3(kLikeBlock), 0, as_stream(stream),
                       reinterpret_cast<const double2*>(htilde), reinterpret_cast<const double2*>(dtilde), n, F, df, f0, partial, nchunks);
    int rc = check_launch("fd_likelihood_partial");
    if (rc) return rc;
    hipLaunchKernelGGL(k_fd_likelihood_final, dim3(n), dim3(64), 0, as_stream(stream), partial, n, nchunks, df, logl);
    return check_launch("fd_likelihood_final");
}

size_t eobhip_fd_likelihood_partial_doubles(int n, int F) {
    const int per = kLikeBlock * kLikePerThread;
    return (size_t)n * (size_t)((F + per - 1) / per);
}

}  // extern "C"

// ---------------------------------------------- likelihood without allocation
// The partial sums of eobhip_fd_likelihood_static live in file-scope device
// memory: one copy per GPU, held until the process ends.  Host code reaches a
// GPU's copy only through the address hipGetSymbolAddress returns with that GPU
// current (the array's name is a host-side stand-in, not a device address).
namespace fdlik_static {
constexpr size_t kScratchDoubles = size_t(1) << 19;   // 4 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];
constexpr int kMaxDevices = 64;
static std::mutex g_lock;
static double* g_ptr[kMaxDevices] = {};

// this GPU's copy of `scratch`, looked up on the first call on the device
static int scratch_ptr(double** out) {
    int dev = -1;
    int rc = hip_status(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("fd_likelihood_static: device %d outside the %d devices the library tracks", dev, kMaxDevices);
        return EOBHIP_EINVAL;
    }
    std::lock_guard<std::mutex> g(g_lock);
    if (!g_ptr[dev]) {
        void* p = nullptr;
        rc = hip_status(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (rc) return rc;
        g_ptr[dev] = static_cast<double*>(p);
    }
    *out = g_ptr[dev];
    return EOBHIP_OK;
}
}  // namespace fdlik_static

extern "C" {

size_t eobhip_fd_likelihood_static_max_partials(void) { return fdlik_static::kScratchDoubles; }

int eobhip_fd_likelihood_static(const double* htilde, const double* dtilde, int n, int F, double df, double f0, double* logl,
                                void* stream) {
    EOBHIP_REQUIRE(n >= 1 && F >= 1, "bad sizes");
    const size_t need = eobhip_fd_likelihood_partial_doubles(n, F);
    EOBHIP_REQUIRE(need <= fdlik_static::kScratchDoubles,
                   "fd_likelihood_static: %zu partial sums (n = %d, F = %d) exceed the library's static buffer of %zu; "
                   "use eobhip_fd_likelihood with a caller-provided buffer",
                   need, n, F, fdlik_static::kScratchDoubles);
    double* partial = nullptr;
    const int rc = fdlik_static::scratch_ptr(&partial);
    if (rc) return rc;
    // every (binary, chunk) partial is written before it is read: nothing to clear
    return eobhip_fd_likelihood(htilde, dtilde, partial, n, F, df, f0, logl, stream);
}

}  // extern "C"
