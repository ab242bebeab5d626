// Real-to-complex FFTs of power-of-two length in FP64 for batches of rows.
//
// A row of N real samples is taken as H = N/2 complex points z_j = x_2j + i
// x_2j+1; with Z their transform, X_k = E_k - i W_N^k O_k for k <= H, where
// E_k = (Z_k + conj Z_{H-k})/2, O_k = (Z_k - conj Z_{H-k})/2 and W_N = e^{-2 pi i/N}.
//
// What bounds it is memory, so the design counts passes over it.  A block of
// kFftThreads threads holds kFftPoints complex points, 16 per thread in
// registers, and exchanges them through LDS between radix-16 stages (real
// parts first, then imaginary parts, so that the exchange buffer is 8 bytes
// per point and two blocks share a CU's LDS; but for the column pass of 2^15,
// whose 64 columns' step table makes it 87 kB and one block a CU):
//   H <= kFftPoints   one kernel (k_rfft_one): whole rows in a block;
//   larger H = A B    two kernels, the row as an A x B matrix (j = a B + b):
//     k_rfft_cols: length-A transforms of C consecutive columns b, times
//                  W_H^(b ka), stored transposed at b A + ka;
//     k_rfft_rows: length-B transforms over b for C consecutive ka and their
//                  C partners A - ka, which together hold k = ka + A kb and
//                  H - k, so X follows in the block.  It reads and writes the
//                  same index set {q A + ka}, so the output row itself is the
//                  only intermediate and no workspace is needed.
// A batch too small to fill the chip is bound by one block's latency: its blocks are
// smaller (a wavefront for rows of 2^10 and 2^11, 128 threads for the two kernels,
// which also take rows of 2^14 then).  us, with blocks of kFftThreads for every batch,
// now, and hipFFT's plan: one row of 2^11 9.4, 6.1, 7.2, of 2^14 12.2, 9.4, 11.8, of
// 2^15 15.0, 10.1, 12.9, of 2^18 17.9, 11.9, 16.4; 32 rows of 2^11 10.3, 6.3, 6.5; up
// to 64 rows of 2^10 9.0, 5.8, 5.5.
// Measured on 256 rows of 2^20 samples: 1.77 ms, the two passes at 4.85 TB/s
// (a large copy reaches 4.97) against 4.62 ms for hipFFT's plan (three
// transposes, two transforms and the real step); 4096 rows of 2^10: 20 us
// against 370.  Relative error against extended precision 3.1e-16 at 2^20
// (hipFFT's 5.6e-16): twiddles are table entries from sincospi, products of
// two at most.
// Stages are Stockham's (self-sorting): thread p of a transform of length n
// holds points p + (n/16) u, u < 16, when a stage starts and after the last.
#pragma once
#include <hip/hip_runtime.h>

#include "eobhip_common.hpp"

namespace eobhip_detail {

constexpr int kFftThreads = 512;   // the most
constexpr int kFftPoints = 16 * kFftThreads;
constexpr int kFftMinLog2 = kRfftMinLog2, kFftMaxLog2 = kRfftMaxLog2;   // N
constexpr int kFftOneMaxLog2 = kRfftOneMaxLog2;   // N whose H = N/2 points fit one block
static_assert((1 << (kFftOneMaxLog2 - 1)) == kFftPoints, "one-kernel limit");

__device__ __forceinline__ double2 cmul2(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

// e^{-2 pi i x}
__device__ __forceinline__ double2 fft_unit(double x) {
    double s, c;
    sincospi(-2.0 * x, &s, &c);
    return make_double2(c, s);
}

// ---------------------------------------------------------------- butterflies
// forward transforms in registers of the R values v[o], v[o + st], ...
__device__ __forceinline__ void bfly4(double2& a, double2& b, double2& c, double2& d) {
    const double2 s = make_double2(a.x + c.x, a.y + c.y), t = make_double2(a.x - c.x, a.y - c.y);
    const double2 u = make_double2(b.x + d.x, b.y + d.y), w = make_double2(b.x - d.x, b.y - d.y);
    a = make_double2(s.x + u.x, s.y + u.y);
    c = make_double2(s.x - u.x, s.y - u.y);
    b = make_double2(t.x + w.y, t.y - w.x);   // t - i w
    d = make_double2(t.x - w.y, t.y + w.x);   // t + i w
}

constexpr double kC16_1 = 0.92387953251128675613, kS16_1 = 0.38268343236508977173;   // cos, sin(pi/8)
constexpr double kC8 = 0.70710678118654752440;

// times W_16^k, k known at compile time
template <int K>
__device__ __forceinline__ double2 mul_w16(double2 a) {
    if constexpr (K == 0) return a;
    else if constexpr (K == 1) return make_double2(a.x * kC16_1 + a.y * kS16_1, a.y * kC16_1 - a.x * kS16_1);
    else if constexpr (K == 2) return make_double2((a.x + a.y) * kC8, (a.y - a.x) * kC8);
    else if constexpr (K == 3) return make_double2(a.x * kS16_1 + a.y * kC16_1, a.y * kS16_1 - a.x * kC16_1);
    else if constexpr (K == 4) return make_double2(a.y, -a.x);
    else if constexpr (K == 6) return make_double2((a.y - a.x) * kC8, -(a.x + a.y) * kC8);
    else {
        static_assert(K == 9, "radix-16 twiddles");
        return make_double2(-(a.x * kC16_1 + a.y * kS16_1), a.x * kS16_1 - a.y * kC16_1);
    }
}

// radix-R transform of v[o + st q], q < R, result in place (R = 2, 4, 8, 16)
template <int R>
__device__ __forceinline__ void bfly(double2 (&v)[16], int o) {
    constexpr int st = 16 / R;
    if constexpr (R == 2) {
        const double2 a = v[o], b = v[o + st];
        v[o] = make_double2(a.x + b.x, a.y + b.y);
        v[o + st] = make_double2(a.x - b.x, a.y - b.y);
    } else if constexpr (R == 4) {
        bfly4(v[o], v[o + st], v[o + 2 * st], v[o + 3 * st]);
    } else if constexpr (R == 8) {
        // n = 4 a + b, k = c + 2 d
        double2 t[8];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const double2 x = v[o + st * b], y = v[o + st * (b + 4)];
            t[b] = make_double2(x.x + y.x, x.y + y.y);
            t[4 + b] = make_double2(x.x - y.x, x.y - y.y);
        }
        t[5] = mul_w16<2>(t[5]);
        t[6] = mul_w16<4>(t[6]);
        t[7] = mul_w16<6>(t[7]);
        bfly4(t[0], t[1], t[2], t[3]);
        bfly4(t[4], t[5], t[6], t[7]);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            v[o + st * (2 * d)] = t[d];
            v[o + st * (2 * d + 1)] = t[4 + d];
        }
    } else {
        static_assert(R == 16, "radix 2, 4, 8 or 16");
        // n = 4 a + b, k = c + 4 d
#pragma unroll
        for (int b = 0; b < 4; ++b) bfly4(v[b], v[b + 4], v[b + 8], v[b + 12]);
        // now v[b + 4 c] = t_c[b]
        v[5] = mul_w16<1>(v[5]);
        v[6] = mul_w16<2>(v[6]);
        v[7] = mul_w16<3>(v[7]);
        v[9] = mul_w16<2>(v[9]);
        v[10] = mul_w16<4>(v[10]);
        v[11] = mul_w16<6>(v[11]);
        v[13] = mul_w16<3>(v[13]);
        v[14] = mul_w16<6>(v[14]);
        v[15] = mul_w16<9>(v[15]);
        double2 t[16];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            bfly4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
#pragma unroll
            for (int d = 0; d < 4; ++d) t[c + 4 * d] = v[4 * c + d];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = t[k];
    }
}

// ----------------------------------------------------------------- exchanges
// 16 values per thread: value u goes to w(u), then value u comes from r(u);
// real parts, then imaginary parts, through the same buffer.  Every thread of
// the block calls it; it ends with the reads done (the caller synchronises
// before the buffer is written again).
template <class W, class R>
__device__ __forceinline__ void lds_exchange(double2 (&v)[16], double* buf, const W& w, const R& r) {
#pragma unroll
    for (int u = 0; u < 16; ++u) buf[w(u)] = v[u].x;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u].x = buf[r(u)];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) buf[w(u)] = v[u].y;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u].y = buf[r(u)];
}

// Stockham positions: outputs of butterfly j of a radix-16 stage with S done
// (the product of the earlier radices), and a stage's inputs
__device__ __forceinline__ int stage_out(int j, int S, int q) { return (j / S) * S * 16 + (j % S) + q * S; }

// W_n^e from a table of half a circle (entries e < n/2)
struct HalfTable {
    const double2* t;
    int n;
    __device__ __forceinline__ double2 operator()(int e) const {
        const int h = n >> 1;
        const double2 w = t[e & (h - 1)];
        return (e & h) ? make_double2(-w.x, -w.y) : w;
    }
};
// W_n^e as a product of two table entries (hi: W_n^(64 e1), lo: W_n^e0)
struct SplitTable {
    const double2 *hi, *lo;
    __device__ __forceinline__ double2 operator()(int e) const { return cmul2(hi[e >> 6], lo[e & 63]); }
};

// twiddles of a radix-R stage with S = 2^LS done in a transform of length
// 2^LN: input q of butterfly j times W_{SR}^{(j mod S) q}; butterflies j = p + (n/16) m
template <int LN, int LS, int R, class T>
__device__ __forceinline__ void stage_twiddle(double2 (&v)[16], int p, const T& tw) {
    constexpr int st = 16 / R, S = 1 << LS, scale = (1 << LN) / (S * R);
#pragma unroll
    for (int m = 0; m < st; ++m) {
        const int j = (p + ((1 << LN) / 16) * m) & (S - 1);
#pragma unroll
        for (int q = 1; q < R; ++q) v[m + st * q] = cmul2(v[m + st * q], tw(scale * j * q));
    }
}

template <int R>
__device__ __forceinline__ void stage_bfly(double2 (&v)[16]) {
#pragma unroll
    for (int m = 0; m < 16 / R; ++m) bfly<R>(v, m);
}

// The stages of a length-2^LN transform (LN = 6 .. 13) whose points are in v
// (point p + (n/16) u in slot u).  addr(pos) places a point of this thread's
// transform in the exchange buffer; before the last stage the thread may turn
// to point p2 of another transform of the block, placed by addr2 (the same
// placement at the end of the write: the last exchange writes with addr2w and
// reads with addr2r).
template <int LN, class T, class A, class AW, class AR>
__device__ __forceinline__ void fft_stages(double2 (&v)[16], int p, int p2, double* buf, const T& tw, const A& addr, const AW& last_w,
                                           const AR& last_r) {
    constexpr int q16 = (1 << LN) / 16;
    constexpr int full = (LN % 4 == 0) ? LN / 4 : LN / 4 + 1;   // stages
    constexpr int RL = (LN % 4 == 0) ? 16 : (1 << (LN % 4));    // last radix
    static_assert(full >= 2 && full <= 4, "5 <= LN <= 13");
    bfly<16>(v, 0);
    if constexpr (full > 2) {
        lds_exchange(v, buf, [&](int u) { return addr(stage_out(p, 1, u)); }, [&](int u) { return addr(p + q16 * u); });
        __syncthreads();
        stage_twiddle<LN, 4, 16>(v, p, tw);
        bfly<16>(v, 0);
    }
    if constexpr (full > 3) {
        lds_exchange(v, buf, [&](int u) { return addr(stage_out(p, 16, u)); }, [&](int u) { return addr(p + q16 * u); });
        __syncthreads();
        stage_twiddle<LN, 8, 16>(v, p, tw);
        bfly<16>(v, 0);
    }
    constexpr int LS = 4 * (full - 1), SP = 1 << (4 * (full - 2));   // done before the last stage, and before the one just run
    lds_exchange(v, buf, [&](int u) { return last_w(stage_out(p, SP, u)); }, [&](int u) { return last_r(p2 + q16 * u); });
    stage_twiddle<LN, LS, RL>(v, p2, tw);
    stage_bfly<RL>(v);
}

// X_k from Z_k, Z_{H-k} and W_N^k
__device__ __forceinline__ double2 real_bin(double2 z, double2 zp, double2 w) {
    const double er = 0.5 * (z.x + zp.x), ei = 0.5 * (z.y - zp.y);
    const double dr = 0.5 * (z.x - zp.x), di = 0.5 * (z.y + zp.y);
    // -i W O
    return make_double2(er + (w.x * di + w.y * dr), ei - (w.x * dr - w.y * di));
}

// W_32^u, u < 16
__device__ __forceinline__ double2 w32(int u) {
    constexpr double c[17] = {1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708, 0.70710678118654752440,
                              0.55557023301960222474, 0.38268343236508977173, 0.19509032201612826785, 0.0, -0.19509032201612826785,
                              -0.38268343236508977173, -0.55557023301960222474, -0.70710678118654752440, -0.83146961230254523708,
                              -0.92387953251128675613, -0.98078528040323044913, -1.0};
    return make_double2(c[u], u <= 8 ? -c[8 - u] : -c[u - 8]);
}

// X_k for this thread's 16 points k, each with its partner Z_{H-k}, which the
// block holds: slot u of the thread pairs with slot 15 - u of thread `mate`
// (or, where `self0`, with its own slot 16 - u, slots 0 and 8 with themselves).
// Half the slots go through LDS at a time as whole complex values, so that no
// second set of 16 is held in registers.  w0 is W_N^k of slot 0; use(u, X).
template <int T, class Use>
__device__ __forceinline__ void real_bins(const double2 (&v)[16], double* buf, int mate, bool self0, double2 w0, const Use& use) {
    double2* half = reinterpret_cast<double2*>(buf);   // 8 values per thread
    __syncthreads();
#pragma unroll
    for (int u = 8; u < 16; ++u) half[(u - 8) * T + threadIdx.x] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        double2 zp = half[((self0 && u > 0) ? 8 - u : 7 - u) * T + mate];
        if (u == 0) zp = make_double2(self0 ? v[0].x : zp.x, self0 ? v[0].y : zp.y);
        use(u, real_bin(v[u], zp, cmul2(w0, w32(u))));
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) half[u * T + threadIdx.x] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 8; u < 16; ++u) {
        double2 zp = half[((self0 && u > 8) ? 16 - u : 15 - u) * T + mate];
        if (u == 8) zp = make_double2(self0 ? v[8].x : zp.x, self0 ? v[8].y : zp.y);
        use(u, real_bin(v[u], zp, cmul2(w0, w32(u))));
    }
}

// sum of |X_k|^2 w_k over the bins this thread's first 8 points give, k and H - k
// of each pair from one (E, T): X_k = E + T, X_{H-k} = conj(E - T).  Every pair
// of the block is some thread's (a thread's slots 8 .. 15 are its mates'), the
// Nyquist bin is k = 0's partner, and slot 8 of `self0` is its own partner,
// X = conj Z.  Half the exchange and products of real_bins.  weight(u) and
// mirror(u): w at slot u's k and at H - k.
template <int T, class Wt, class Mi>
__device__ __forceinline__ double real_norms(const double2 (&v)[16], double* buf, int mate, bool self0, double2 w0, const Wt& weight,
                                             const Mi& mirror) {
    double2* half = reinterpret_cast<double2*>(buf);
    double wk[8], wm[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        wk[u] = weight(u);
        wm[u] = mirror(u);
    }
    __syncthreads();
#pragma unroll
    for (int u = 8; u < 16; ++u) half[(u - 8) * T + threadIdx.x] = v[u];
    __syncthreads();
    double acc = self0 ? (v[8].x * v[8].x + v[8].y * v[8].y) * weight(8) : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        double2 zp = half[((self0 && u > 0) ? 8 - u : 7 - u) * T + mate];
        if (u == 0) zp = make_double2(self0 ? v[0].x : zp.x, self0 ? v[0].y : zp.y);
        const double2 z = v[u], w = cmul2(w0, w32(u));
        const double er = 0.5 * (z.x + zp.x), ei = 0.5 * (z.y - zp.y);
        const double dr = 0.5 * (z.x - zp.x), di = 0.5 * (z.y + zp.y);
        const double tr = w.x * di + w.y * dr, ti = -(w.x * dr - w.y * di);
        const double ar = er + tr, ai = ei + ti, br = er - tr, bi = ei - ti;
        acc += (ar * ar + ai * ai) * wk[u];
        acc += (br * br + bi * bi) * wm[u];
    }
    return acc;
}

// Consecutive work on one XCD: block i runs on XCD i mod 8, and neighbouring
// work items share cache lines (rows start at any 16-byte boundary), so each
// XCD takes a contiguous run of them.
__device__ __forceinline__ unsigned xcd_run(unsigned bid, unsigned nblk) {
    const unsigned x = bid & 7, q = nblk >> 3, rem = nblk & 7;
    return x * q + (x < rem ? x : rem) + (bid >> 3);
}

}  // namespace eobhip_detail
