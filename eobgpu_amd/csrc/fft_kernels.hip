// Batched real-to-complex FFTs (see fft.hpp) and the weighted norm of the
// transforms that the support-length likelihood needs, computed in the last
// pass so that those transforms are never written.
#include <hip/hip_runtime.h>

#include "eobhip_common.hpp"
#include "fft.hpp"

using namespace eobhip_detail;

namespace {

// Where a pass of a batch of rows finds its input and leaves its output.
// in: rows of N doubles (stride in_stride doubles); out: rows of complex bins
// (stride out_stride).  nvalid (optional): samples of the row that are not
// zero by definition, count[map[first + row]]; the rest are not read.
struct Rows {
    const double* in;
    double2* out;
    long long in_stride, out_stride;
    const int* count;
    const long long* map;
    int rows;
};

// Sum of |X_k|^2 w_k instead of the bins: w (stride 1) and one partial per
// (row, block of the row), partial[map[row] * pstride + block].
struct Norm {
    const double* w;
    double* partial;
    int pstride;
};

__device__ __forceinline__ long long valid_samples(const Rows& a, int row, long long N) {
    if (!a.count) return N;
    const long long c = a.count[a.map[row]];
    return c < 0 ? 0 : (c > N ? N : c);
}

// the two real samples of point j, zero past the row's samples (the caller
// keeps samples up to the next even count defined)
__device__ __forceinline__ double2 load_point(const double2* __restrict__ z, long long j, long long nv) {
    return 2 * j < nv ? z[j] : make_double2(0.0, 0.0);
}

// Sum of a value over the block's threads with the same (threadIdx.x / G); G a
// power of two.  The result is valid on the first thread of each G.
template <int G>
__device__ __forceinline__ double group_sum(double v, double* red) {
    constexpr int W = G < 64 ? G : 64;
#pragma unroll
    for (int off = W / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if constexpr (G > 64) {
        __syncthreads();
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x % G == 0) {
            v = 0.0;
            for (int k = 0; k < G / 64; ++k) v += red[(threadIdx.x >> 6) + k];
        }
    }
    return v;
}

// ------------------------------------------------------------ whole rows
// H = 2^LH points per row, kFftPoints / H rows per block.  Twiddles of up to
// 8192 points are products of two small tables.
template <int LH, bool kNorm, int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T == kFftThreads ? 4 : 2))) void k_rfft_one(Rows a, Norm nm) {
    constexpr int H = 1 << LH, per = H / 16;   // threads per row
    __shared__ double buf[17 * T];
    __shared__ double2 hi[H / 64], lo[64];
    const int t = threadIdx.x, rr = t / per, p = t % per;
    const long long row = (long long)blockIdx.x * (blockDim.x / per) + rr;
    const bool on = row < a.rows;
    const double2* z = reinterpret_cast<const double2*>(a.in + (on ? row : 0) * a.in_stride);
    const long long nv = on ? valid_samples(a, (int)row, 2LL * H) : 0;
    double2 v[16];   // on their way while the tables are made
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = load_point(z, p + per * u, nv);
    for (int i = t; i < H / 64; i += blockDim.x) hi[i] = fft_unit((double)i * (64.0 / H));
    if (t < 64) lo[t] = fft_unit((double)t * (1.0 / H));
    double2 w0;
    if constexpr (!kNorm) w0 = fft_unit((double)p * (0.5 / H));
    const auto addr = [&](int pos) { return rr * (H + H / 16) + pos + (pos >> 4); };
    const SplitTable tw{hi, lo};
    fft_stages<LH>(v, p, p, buf, tw, addr, addr, addr);
    const int mate = rr * per + ((per - p) & (per - 1));
    if constexpr (kNorm) {
        w0 = fft_unit((double)p * (0.5 / H));
        const double acc = real_norms<T>(v, buf, mate, p == 0, w0, [&](int u) { return nm.w[p + per * u]; },
                                      [&](int u) { return nm.w[H - (p + per * u)]; });
        const double s = group_sum<per>(acc, buf);   // the first barrier inside is after every thread's reads of buf
        if (p == 0 && on) nm.partial[a.map[row] * nm.pstride] = s;
    } else {
        real_bins<T>(v, buf, mate, p == 0, w0, [&](int u, double2 x) {
            if (on) a.out[row * a.out_stride + p + per * u] = x;
        });
        if (p == 0 && on) a.out[row * a.out_stride + H] = make_double2(v[0].x - v[0].y, 0.0);   // X_H
    }
}

// --------------------------------------------------- columns of an A x B row
template <int LA, int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T == kFftThreads ? 4 : 2))) void k_rfft_cols(Rows a, int LB) {
    constexpr int A = 1 << LA, C = 16 * T / A, per = A / 16;
    constexpr int pad = C >= 32 ? 1 : 32 / C;
    constexpr int skew = T;
    constexpr int kWords = 16 * T + (skew > C * pad ? skew : C * pad);
    __shared__ double buf[kWords];
    __shared__ double2 tab[A / 2], step[C][16];
    const int B = 1 << LB, t = threadIdx.x;
    const unsigned id = xcd_run(blockIdx.x, gridDim.x);
    const int groups = B / C;
    const int row = (int)(id / groups), b0 = (int)(id % groups) * C;
    const long long N = 2LL * A * B;
    const double invH = 2.0 / (double)N;
    const int i = t % C, p = t / C;
    const double2* z = reinterpret_cast<const double2*>(a.in + row * a.in_stride);
    const long long nv = valid_samples(a, row, N);
    double2 v[16];   // on their way while the tables are made
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = load_point(z, ((long long)(p + per * u) << LB) + b0 + i, nv);
    for (int e = t; e < A / 2; e += T) tab[e] = fft_unit((double)e * (1.0 / A));
    // W_H^(b (A/16) u): the between-pass twiddle's step along a thread's outputs
    for (int e = t; e < C * 16; e += T) {
        const int u = e & 15, i = e >> 4;
        step[i][u] = fft_unit((double)((long long)(b0 + i) * u) * ((double)per * invH));
    }
    // column fastest until the last exchange, which turns to position fastest
    // (a column's outputs are stored contiguously)
    const int i2 = t / per, p2 = t % per;
    const HalfTable tw{tab, A};
    fft_stages<LA>(v, p, p2, buf, tw, [&](int pos) { return (pos + (pos >> 4)) * C + i; }, [&](int pos) { return i * (A + pad) + pos; },
                   [&](int pos) { return i2 * (A + pad) + pos; });
    const long long b = b0 + i2;
    const double2 w0 = fft_unit((double)(b * p2) * invH);
    double2* o = a.out + row * a.out_stride + (b << LA);
#pragma unroll
    for (int u = 0; u < 16; ++u) o[p2 + per * u] = cmul2(v[u], cmul2(w0, step[i2][u]));
}

// ------------------------------------------------------ rows of an A x B row
template <int LB, bool kNorm, int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T == kFftThreads ? 4 : 2))) void k_rfft_rows(Rows a, Norm nm, int LA) {
    constexpr int B = 1 << LB, C2 = 16 * T / B, C = C2 / 2, per = B / 16;
    __shared__ double buf[17 * T];
    __shared__ double2 tab[B / 2];
    const int A = 1 << LA, t = threadIdx.x;
    const unsigned id = xcd_run(blockIdx.x, gridDim.x);
    const int groups = A / C2;
    const int row = (int)(id / groups), g = (int)(id % groups);
    const long long H = (long long)A * B;
    // (the tables after the loads have been issued hide a small batch's latency and cost the
    // large blocks registers)
    const auto tables = [&] {
        for (int e = t; e < B / 2; e += T) tab[e] = fft_unit((double)e * (1.0 / B));
    };
    if constexpr (T == kFftThreads) tables();
    const int i = t % C2, p = t / C2;
    // slots i < C: ka = g C + i; the others their partners A - ka (ka = A/2 in the place of 0's)
    const int kl = g * C + (i & (C - 1));
    const int ka = i < C ? kl : (kl == 0 ? A / 2 : A - kl);
    // a row is at most 16 MiB + 16 bytes: 32-bit byte offsets from its (uniform) start
    char* o = reinterpret_cast<char*>(a.out + row * a.out_stride);
    const unsigned at = ((unsigned)ka + ((unsigned)p << LA)) * 16u, up = (unsigned)(per << LA) * 16u;
    double2 v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = *reinterpret_cast<const double2*>(o + (at + up * u));
    if constexpr (T != kFftThreads) tables();
    const HalfTable tw{tab, B};
    const auto addr = [&](int pos) { return (pos + (pos >> 4)) * C2 + i; };
    fft_stages<LB>(v, p, p, buf, tw, addr, addr, addr);
    // the partner H - k of k = ka + A kb: row A - ka, kb' = B - 1 - kb; rows 0
    // (kb' = B - kb) and A/2 are their own
    const int mate = (kl == 0 ? i : (i ^ C)) + C2 * (((ka == 0 ? per : per - 1) - p) & (per - 1));
    const double2 w0 = fft_unit((double)(ka + (long long)p * A) * (0.5 / (double)H));
    const bool self0 = ka == 0 && p == 0;
    if constexpr (kNorm) {
        const double* w = nm.w;
        const unsigned k0 = (unsigned)ka + ((unsigned)p << LA), up = (unsigned)(per << LA);
        const double acc = real_norms<T>(v, buf, mate, self0, w0, [&](int u) { return w[k0 + up * u]; },
                                      [&](int u) { return w[(unsigned)H - (k0 + up * u)]; });
        static_assert(T == kFftThreads, "rfft_norm_partials counts these blocks");
        const double s = group_sum<T>(acc, buf);
        if (t == 0) nm.partial[a.map[row] * nm.pstride + g] = s;
    } else {
        real_bins<T>(v, buf, mate, self0, w0, [&](int u, double2 x) { *reinterpret_cast<double2*>(o + (at + up * u)) = x; });
        if (self0) *reinterpret_cast<double2*>(o + 16 * H) = make_double2(v[0].x - v[0].y, 0.0);   // X_H
    }
}

// A of H = A B for H > kFftPoints: the larger half
int log2_cols(int lh) { return (lh + 1) / 2; }

template <bool kNorm, int T>
int launch_two(const Rows& a, const Norm& nm, int lh, hipStream_t st) {
    constexpr int lp = T == 512 ? 13 : 11;   // points of a block
    static_assert(16 * T == 1 << lp);
    const int la = log2_cols(lh), lb = lh - la;
    const long long nc = (long long)a.rows << (lh - lp);
    EOBHIP_REQUIRE(nc < (1LL << 31), "rfft: too many rows");
    const dim3 grid((unsigned)nc);
    switch (la) {
#define EOBHIP_COLS(L) \
    case L: hipLaunchKernelGGL((k_rfft_cols<L, T>), grid, dim3(T), 0, st, a, lb); break;
        EOBHIP_COLS(7) EOBHIP_COLS(8) EOBHIP_COLS(9) EOBHIP_COLS(10)
#undef EOBHIP_COLS
        default: set_error("rfft: unsupported length 2^%d", lh + 1); return EOBHIP_EINVAL;
    }
    int rc = check_launch("rfft columns");
    if (rc) return rc;
    switch (lb) {
#define EOBHIP_ROWS(L) \
    case L: hipLaunchKernelGGL((k_rfft_rows<L, kNorm, T>), grid, dim3(T), 0, st, a, nm, la); break;
        EOBHIP_ROWS(7) EOBHIP_ROWS(8) EOBHIP_ROWS(9) EOBHIP_ROWS(10)
#undef EOBHIP_ROWS
        case 6:   // 2^14, small blocks only
            if constexpr (T < kFftThreads) {
                hipLaunchKernelGGL((k_rfft_rows<6, kNorm, T>), grid, dim3(T), 0, st, a, nm, la);
                break;
            }
            [[fallthrough]];
        default: set_error("rfft: unsupported length 2^%d", lh + 1); return EOBHIP_EINVAL;
    }
    return check_launch("rfft rows");
}

template <bool kNorm>
int launch_rows(const Rows& a, const Norm& nm, int LN, hipStream_t st) {
    const int lh = LN - 1;
    // small blocks in two passes where kFftThreads of them would leave CUs idle (rows of
    // 2^14: up to 31, 9.6 us for 12.5 in one pass; 32 rows 12.7 in one)
    if constexpr (!kNorm)
        if (LN >= kFftOneMaxLog2 && (long long)a.rows << lh < (LN == kFftOneMaxLog2 ? 32LL : 256LL) << 13) return launch_two<kNorm, 128>(a, nm, lh, st);
    if (LN <= kFftOneMaxLog2) {
        // threads: as many rows a block as leave the batch a block per CU, at least one row and a wavefront
        int rows = kFftPoints >> lh;
        while (rows > 1 && blocks_for(a.rows, rows) < 256) rows /= 2;
        const int threads = rows << (lh - 4) < 64 ? 64 : rows << (lh - 4);
        const dim3 grid(blocks_for(a.rows, threads >> (lh - 4))), block(threads);
        switch (lh) {
#define EOBHIP_ONE(L) \
    case L: \
        if constexpr (!kNorm && L <= 10) \
            if (threads == 64) { \
                hipLaunchKernelGGL((k_rfft_one<L, kNorm, 64>), grid, block, 0, st, a, nm); \
                break; \
            } \
        hipLaunchKernelGGL((k_rfft_one<L, kNorm, kFftThreads>), grid, block, 0, st, a, nm); \
        break;
            EOBHIP_ONE(9) EOBHIP_ONE(10) EOBHIP_ONE(11) EOBHIP_ONE(12) EOBHIP_ONE(13)
#undef EOBHIP_ONE
            default: set_error("rfft: unsupported length 2^%d", LN); return EOBHIP_EINVAL;
        }
        return check_launch("rfft");
    }
    return launch_two<kNorm, kFftThreads>(a, nm, lh, st);
}

}  // namespace

namespace eobhip_detail {

int rfft_own_log2(const void* in, const void* out, int n, int N) {
    if (n < 1 || N < (1 << kFftMinLog2) || N > (1 << kFftMaxLog2) || (N & (N - 1))) return 0;
    const uintptr_t a = reinterpret_cast<uintptr_t>(in), b = reinterpret_cast<uintptr_t>(out);
    if ((a | b) & 15) return 0;
    const uintptr_t na = (uintptr_t)n * N * 8, nb = (uintptr_t)n * (N / 2 + 1) * 16;
    if (a < b + nb && b < a + na) return 0;
    return __builtin_ctz((unsigned)N);
}

int rfft_weighted_norm(const double* in, long long in_stride, double* work, int n, int log2N, const int* count, const long long* map,
                       const double* w, double* partial, int pstride, hipStream_t st) {
    return launch_rows<true>(Rows{in, reinterpret_cast<double2*>(work), in_stride, 1LL << (log2N - 1), count, map, n}, Norm{w, partial, pstride},
                             log2N, st);
}

int rfft_own(const double* in, double* out, int n, int log2N, hipStream_t st) {
    const long long N = 1LL << log2N;
    return launch_rows<false>(Rows{in, reinterpret_cast<double2*>(out), N, N / 2 + 1, nullptr, nullptr, n}, Norm{nullptr, nullptr, 0}, log2N,
                              st);
}

}  // namespace eobhip_detail
