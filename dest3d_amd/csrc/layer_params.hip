// The small parameters of a decoder layer in the form its kernels read (gfx950): every array converted to fp32 and laid one
// behind the other, and A[h][n] = -exp(A_log[h]) for all state columns (models/dest_module.py:485-500, :562).
// A few thousand values: the launch is all it costs.  As tensor operators it was six launches (concatenation, conversion, exp,
// negation, expansion of A, conversion of D), 25 - 30 us of host time a layer where a forward layer of one scene runs at the
// pace of its launches.
// Compiled without -ffast-math: exp must be the accurate one.
#include "issm_dev.h"

namespace issm {

__global__ __launch_bounds__(NTHREADS) void k_layer_params(LayerParamsP p) {
  const int e = blockIdx.x * NTHREADS + threadIdx.x;
  if (e < p.total) {
    int s = 0, at = e;
    while (at >= p.n[s]) at -= p.n[s++];   // e < total: ends inside the last array
    p.out[e] = p.bf16[s] ? bf16_to_f(((const uint16_t*)p.src[s])[at]) : ((const float*)p.src[s])[at];
  } else if (e - p.total < p.H * p.K) {
    const int h = (e - p.total) / p.K, s = p.a_log;
    const float v = p.bf16[s] ? bf16_to_f(((const uint16_t*)p.src[s])[h]) : ((const float*)p.src[s])[h];
    p.A[e - p.total] = -expf(v);
  }
}

int launch_layer_params(const LayerParamsP& p, hipStream_t st) {
  const int n = p.total + p.H * p.K;
  hipLaunchKernelGGL(k_layer_params, dim3((n + NTHREADS - 1) / NTHREADS), dim3(NTHREADS), 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
