// One entry of a decoder layer's small parameters (see layer_params.hip); for sources compiled without -ffast-math.
#pragma once
#include "issm_dev.h"

namespace issm {

// (The arrays are chosen by comparisons with constant indexes: an index of its own would take the arguments through scratch memory.)
__device__ __forceinline__ void layer_params_entry(const LayerParamsP& p, int e) {
  const bool in_A = e >= p.total;
  if (in_A && e - p.total >= p.H * p.K) return;
  const int h = in_A ? (e - p.total) / p.K : 0;
  const void* src = p.src[0];
  int bf16 = p.bf16[0], at = in_A ? h : e, first = 0;
#pragma unroll
  for (int i = 1; i < LAYER_ARRAYS; ++i) {
    first += p.n[i - 1];
    const bool here = in_A ? p.a_log == i : e >= first;
    src = here ? p.src[i] : src;
    bf16 = here ? p.bf16[i] : bf16;
    if (!in_A) at = here ? e - first : at;
  }
  const float v = bf16 ? bf16_to_f(((const uint16_t*)src)[at]) : ((const float*)src)[at];
  if (in_A) p.A[e - p.total] = -expf(v);
  else p.out[e] = v;
}

}  // namespace issm
