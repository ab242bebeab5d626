// Host-side plumbing shared by the C-ABI translation units: error reporting and
// launch helpers.  No entry point aborts the process; failures return a status
// and leave a message for eobhip_last_error().
#pragma once
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdarg>
#include "../../include/eobhip.h"

namespace eobhip_detail {

void set_error(const char* fmt, ...);

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return EOBHIP_EHIP;
    }
    return EOBHIP_OK;
}

inline int hip_status(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? EOBHIP_ENOMEM : EOBHIP_EHIP;
    }
    return EOBHIP_OK;
}

inline unsigned blocks_for(long long n, int block) { return (unsigned)((n + block - 1) / block); }

// Row-batched real FFTs through cached hipFFT plans (spline_kernels.hip); rows go
// through in chunks of kFftChunk and then power-of-two chunks.
// inverse = 0: n rows of N doubles -> n rows of N/2+1 complex (D2Z, unnormalised);
// inverse = 1: n rows of N/2+1 complex -> n rows of N doubles (Z2D, unnormalised).
constexpr int kFftChunk = 64;
int fft_exec(int inverse, const void* in, void* out, int rows, int N, void* stream);
int fft_rows(int inverse, const void* in, void* out, int n, int N, void* stream);

// The library's own forward transforms (fft_kernels.hip): log2 N when they take
// these n rows, else 0; and the launch.  They take N = 2^10 .. 2^21 with
// 16-byte aligned rows and an output that does not overlap the input.
int rfft_own_log2(const void* in, const void* out, int n, int N);
int rfft_own(const double* in, double* out, int n, int log2N, hipStream_t st);
constexpr int kRfftMinLog2 = 10, kRfftMaxLog2 = 21;
constexpr int kRfftOneMaxLog2 = 14;   // up to here a block of the most threads holds a row

// sum_k w_k |X_k|^2 over the N/2 + 1 bins of n rows of N samples (same lengths),
// without writing the bins: row r has count[map[r]] samples at in + r in_stride
// (defined up to the next even count, zero after), its rfft_norm_partials(log2 N)
// partial sums go to partial + map[r] pstride.  work: n N/2 complex (unused up
// to N = 2^14).
constexpr __host__ __device__ int rfft_norm_partials(int log2N) { return log2N <= kRfftOneMaxLog2 ? 1 : 1 << (log2N - kRfftOneMaxLog2); }
int rfft_weighted_norm(const double* in, long long in_stride, double* work, int n, int log2N, const int* count, const long long* map,
                       const double* w, double* partial, int pstride, hipStream_t st);

}  // namespace eobhip_detail

#define EOBHIP_REQUIRE(cond, ...)                        \
    do {                                                 \
        if (!(cond)) {                                   \
            eobhip_detail::set_error(__VA_ARGS__);       \
            return EOBHIP_EINVAL;                        \
        }                                                \
    } while (0)
