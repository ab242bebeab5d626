// Host build of the resampling kernels' sine and cosine (eobgpu_amd/csrc/eob_fastmath.hpp),
// every multiply-add written as fma() or left apart, as the device build rounds its own.
#include "../eobgpu_amd/csrc/eob_fastmath.hpp"

extern "C" void probe_sincos_phase(const double* x, double* s, double* c, int n) {
    for (int i = 0; i < n; ++i) eob::sincos_phase(x[i], s[i], c[i]);
}
