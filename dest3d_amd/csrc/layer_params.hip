// The small parameters of a decoder layer in the form its kernels read (gfx950): every array converted to fp32 and laid one
// behind the other, and A[h][n] = -exp(A_log[h]) for all state columns (models/dest_module.py:485-500, :562).
// A few thousand values: the launch is all it costs.  As tensor operators it was six launches (concatenation, conversion, exp,
// negation, expansion of A, conversion of D), 25 - 30 us of host time a layer where a forward layer of one scene runs at the
// pace of its launches.
// Compiled without -ffast-math: exp must be the accurate one.
#include "layer_params.h"
#include "transpose_dev.h"

namespace issm {

__global__ __launch_bounds__(NTHREADS) void k_layer_params(LayerParamsP p) { layer_params_entry(p, blockIdx.x * NTHREADS + threadIdx.x); }

int launch_layer_params(const LayerParamsP& p, hipStream_t st) {
  const int n = p.total + p.H * p.K;
  hipLaunchKernelGGL(k_layer_params, dim3((n + NTHREADS - 1) / NTHREADS), dim3(NTHREADS), 0, st, p);
  return (int)hipGetLastError();
}

// The same and the queries turned into the layout of the scan's states, which is independent of it (a layer with gradients): 4.9 us at
// 288 features and 8 x 256 queries, 4.1 and 4.8 in two launches.
template <bool BF>
__global__ __launch_bounds__(NTHREADS) void k_layer_begin(LayerParamsP p, TrP t, int params) {
  __shared__ float tile[64][65];
  if ((int)blockIdx.x < params) return layer_params_entry(p, blockIdx.x * NTHREADS + threadIdx.x);
  transpose_nth<BF, BF>(t, (int)blockIdx.x - params, tile);
}

int launch_layer_begin(const LayerParamsP& p, const TrP& t, hipStream_t st) {
  const long params = (p.total + (long)p.H * p.K + NTHREADS - 1) / NTHREADS, blocks = params + transpose_tiles(t);
  if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
  if (t.in_dt) hipLaunchKernelGGL(k_layer_begin<true>, dim3((unsigned)blocks), dim3(NTHREADS), 0, st, p, t, (int)params);
  else hipLaunchKernelGGL(k_layer_begin<false>, dim3((unsigned)blocks), dim3(NTHREADS), 0, st, p, t, (int)params);
  return (int)hipGetLastError();
}

}  // namespace issm
