// A tile of the rearrangement of transpose_states.hip, for the kernels that carry one beside their own work.
#pragma once
#include "issm_dev.h"

namespace issm {

// 64 x 64, by a workgroup of NTHREADS
template <bool IN_BF, bool OUT_BF>
__device__ __forceinline__ void transpose_tile(const TrP& p, int c0, int r0, int b, float (&tile)[64][65]) {
  const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
  const long base = (long)b * p.R * p.C;
  // absent elements read the slab's first element and are not stored: no branch around the loads
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = r0 + ly + 4 * i, c = c0 + lx;
    const bool ok = r < p.R && c < p.C;
    const long o = base + (ok ? (long)r * p.C + c : 0);
    v[i] = IN_BF ? bf16_to_f(((const uint16_t*)p.in0)[o]) : ((const float*)p.in0)[o];
  }
  if (p.in1) {  // uniform; one branch around all sixteen loads
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = r0 + ly + 4 * i, c = c0 + lx;
      const bool ok = r < p.R && c < p.C;
      const long o = base + (ok ? (long)r * p.C + c : 0);
      v[i] += IN_BF ? bf16_to_f(((const uint16_t*)p.in1)[o]) : ((const float*)p.in1)[o];
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] *= p.alpha;
#pragma unroll
  for (int i = 0; i < 16; ++i) tile[ly + 4 * i][lx] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = c0 + ly + 4 * i, r = r0 + lx;
    if (c < p.C && r < p.R) {
      const float a = tile[lx][ly + 4 * i];
      const long o = base + (long)c * p.R + r;
      if (OUT_BF) ((uint16_t*)p.out)[o] = f_to_bf16(a);
      else ((float*)p.out)[o] = a;
    }
  }
}

// workgroups of all of them, and the u-th's tile
inline long transpose_tiles(const TrP& t) { return (long)((t.C + 63) / 64) * ((t.R + 63) / 64) * t.B; }
template <bool IN_BF, bool OUT_BF>
__device__ __forceinline__ void transpose_nth(const TrP& t, int u, float (&tile)[64][65]) {
  const int cs = (t.C + 63) / 64, rs = (t.R + 63) / 64;
  transpose_tile<IN_BF, OUT_BF>(t, u % cs * 64, u / cs % rs * 64, u / (cs * rs), tile);
}

}  // namespace issm
