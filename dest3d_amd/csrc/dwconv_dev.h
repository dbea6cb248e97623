// Per-thread parts of the depthwise convolution's forward (dwconv_silu.hip) that the kernel of param_gen.hip shares with it.
#pragma once
#include "issm_dev.h"

namespace issm {

constexpr int DW_TAPS = 7;

template <bool BF>
__device__ __forceinline__ float dw_ld(const void* p, long i) {
  return BF ? bf16_to_f(((const uint16_t*)p)[i]) : ((const float*)p)[i];
}
template <bool BF>
__device__ __forceinline__ void dw_st(void* p, long i, float v) {
  if (BF) ((uint16_t*)p)[i] = f_to_bf16(v); else ((float*)p)[i] = v;
}

// work item -> (b, tile, c), c fastest, for the first `channels` channels
template <int DW_TL>
__device__ __forceinline__ bool dw_item(const DwConvP& p, long id, int channels, int& b, int& l0, int& c) {
  const int ntile = (p.L + DW_TL - 1) / DW_TL;
  if (id >= (long)p.B * ntile * channels) return false;
  c = (int)(id % channels);
  const long r = id / channels;
  l0 = (int)(r % ntile) * DW_TL;
  b = (int)(r / ntile);
  return true;
}

template <bool BF>
__device__ __forceinline__ float dw_round(float v) { return BF ? bf16_to_f(f_to_bf16(v)) : v; }

// output / gradient address of (set s, row, channel c) with or without the channel split
__device__ __forceinline__ long dw_out_off(const DwConvP& p, long row, int c, bool& head) {
  head = p.split <= 0 || c < p.split;
  if (p.split <= 0) return row * p.C + c;
  return head ? row * p.split + c : row * (p.C - p.split) + (c - p.split);
}

// The forward of a chained pair for work item `id`.  ALL: every channel, with `pre` kept for the backward; otherwise the
// channels in front of the split, and `pre` is not written.
template <bool BF, int DW_TL, bool ALL>
__device__ __forceinline__ void dw_chain_fwd(const DwConvP& p, long id) {
  int b, l0, c;
  if (!dw_item<DW_TL>(p, id, ALL ? p.C : p.split, b, l0, c)) return;
  float w[2][DW_TAPS], bias[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + c) * DW_TAPS + j];
    bias[s] = p.bias[(long)s * p.C + c];
  }
  const long ub = (long)b * p.u_bs + c;
  constexpr int W1 = DW_TL + DW_TAPS - 1, W2 = W1 + DW_TAPS - 1;
  float ub_[W2];  // u[l0 - 6 .. l0 + DW_TL + 5]
#pragma unroll
  for (int j = 0; j < W2; ++j) {
    const int l = l0 + j - 6;
    const float v = dw_ld<BF>(p.u, ub + (long)min(max(l, 0), p.L - 1) * p.u_ls);
    ub_[j] = (l >= 0 && l < p.L) ? v : 0.0f;
  }
  float pre0[W1], y0[W1];  // rows l0 - 3 .. l0 + DW_TL + 2
#pragma unroll
  for (int j = 0; j < W1; ++j) {
    const int l = l0 + j - 3;
    float a = bias[0];
#pragma unroll
    for (int t = 0; t < DW_TAPS; ++t) a = fmaf(w[0][t], ub_[j + t], a);
    a = dw_round<BF>(a);
    pre0[j] = a;
    y0[j] = (l >= 0 && l < p.L) ? dw_round<BF>(a * sigmoidf_(a)) : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < DW_TL; ++i) {
    const int l = l0 + i;
    if (l < p.L) {
      float a = bias[1];
#pragma unroll
      for (int t = 0; t < DW_TAPS; ++t) a = fmaf(w[1][t], y0[i + t], a);
      a = dw_round<BF>(a);
      const float y1 = a * sigmoidf_(a);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const long row = ((long)s * p.B + b) * p.L + l;
        if (ALL) dw_st<BF>(p.pre, row * p.C + c, s ? a : pre0[i + 3]);
        bool head;
        const long o = dw_out_off(p, row, c, head);
        dw_st<BF>(head ? p.y : p.y_tail, o, s ? y1 : y0[i + 3]);
      }
    }
  }
}

// Both outputs of a chained pair at one token and channel, as dw_chain_fwd computes them.
template <bool BF>
__device__ __forceinline__ void dw_chain_at(const DwConvP& p, int b, int l, int c, float& out0, float& out1) {
  float w[2][DW_TAPS], bias[2], u[2 * DW_TAPS - 1], y0[DW_TAPS];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + c) * DW_TAPS + j];
    bias[s] = p.bias[(long)s * p.C + c];
  }
#pragma unroll
  for (int j = 0; j < 2 * DW_TAPS - 1; ++j) {
    const int at = l + j - 6;
    const float v = dw_ld<BF>(p.u, (long)b * p.u_bs + c + (long)min(max(at, 0), p.L - 1) * p.u_ls);
    u[j] = (at >= 0 && at < p.L) ? v : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < DW_TAPS; ++j) {
    const int at = l + j - 3;
    float a = bias[0];
#pragma unroll
    for (int t = 0; t < DW_TAPS; ++t) a = fmaf(w[0][t], u[j + t], a);
    a = dw_round<BF>(a);
    y0[j] = (at >= 0 && at < p.L) ? dw_round<BF>(a * sigmoidf_(a)) : 0.0f;
  }
  float a = bias[1];
#pragma unroll
  for (int t = 0; t < DW_TAPS; ++t) a = fmaf(w[1][t], y0[t], a);
  a = dw_round<BF>(a);
  out0 = y0[3];
  out1 = dw_round<BF>(a * sigmoidf_(a));
}

}  // namespace issm
