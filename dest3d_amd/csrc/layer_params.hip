// The small parameters of a decoder layer in the form its kernels read (gfx950): every array converted to fp32 and laid one
// behind the other, and A[h][n] = -exp(A_log[h]) for all state columns (models/dest_module.py:485-500, :562).
// A few thousand values: the launch is all it costs.  As tensor operators it was six launches (concatenation, conversion, exp,
// negation, expansion of A, conversion of D), 25 - 30 us of host time a layer where a forward layer of one scene runs at the
// pace of its launches.
// Compiled without -ffast-math: exp must be the accurate one.
#include "layer_params.h"

namespace issm {

__global__ __launch_bounds__(NTHREADS) void k_layer_params(LayerParamsP p) { layer_params_entry(p, blockIdx.x * NTHREADS + threadIdx.x); }

int launch_layer_params(const LayerParamsP& p, hipStream_t st) {
  const int n = p.total + p.H * p.K;
  hipLaunchKernelGGL(k_layer_params, dim3((n + NTHREADS - 1) / NTHREADS), dim3(NTHREADS), 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
