// What lies between a decoder layer's scan and its output projections where no gradient is asked for (gfx950), bf16, one launch:
//   key    = RMSNorm(bf16(y0 + y1) * silu(z)) * w          a wave a row of the (batch x seqlen, d_inner) scan outputs
//   query  = LayerNorm(bf16((last0 + last1) / 2)^T)         8 queries a workgroup: their d_inner values, fp32 and one per state
//                                                           row, meet in LDS as bf16 (issm_transpose_states' result)
// Each was a launch or two of its own (add, norm, transpose, LayerNorm), 3 to 4 us whatever its size and as much again to issue;
// at one scene (1024 tokens, 256 queries, 288 features) the four took 15 us, this takes 6.  Bound by the launch and
// one trip to memory; 8 queries a workgroup for 32-byte pieces of a state row and still 32 workgroups at one scene.
// The sums and averages are rounded to bf16 as the separate kernels stored them.
#include "issm_dev.h"

namespace issm {

struct __attribute__((packed, aligned(2))) Bf4At {   // four elements at any element offset
  bf4 v;
};
__device__ __forceinline__ f4 ld_bf4(const uint16_t* p) { return __builtin_convertvector(((const Bf4At*)p)->v, f4); }
__device__ __forceinline__ f4 round_bf4(f4 v) { return __builtin_convertvector(__builtin_convertvector(v, bf4), f4); }
__device__ __forceinline__ void st_bf4(uint16_t* p, f4 v) { ((Bf4At*)p)->v = __builtin_convertvector(v, bf4); }
__device__ __forceinline__ float sum4(f4 v) { return (v[0] + v[1]) + (v[2] + v[3]); }
__device__ __forceinline__ float wave_total(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int LO_Q = 8;   // queries a workgroup

template <int NV>
__global__ __launch_bounds__(NTHREADS) void k_layer_out(LayerOutP p) {
  __shared__ uint16_t tile[LO_Q * (NV * 256 + 4)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, di = p.di;
  if ((int)blockIdx.x < p.key_blocks) {
    const long row = (long)blockIdx.x * 4 + w;
    if (row >= p.rows) return;
    f4 x[NV], z[NV], g[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      x[v] = z[v] = g[v] = zero;
      if (c < di) {
        x[v] = ld_bf4(p.y0 + row * di + c) + ld_bf4(p.y1 + row * di + c);
        z[v] = ld_bf4(p.z + row * p.zs + c);
        g[v] = ld_bf4(p.kw + c);
      }
    }
    float ss = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      x[v] = round_bf4(x[v]);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[v][r] *= z[v][r] * sigmoidf_(z[v][r]);
      ss += sum4(x[v] * x[v]);
    }
    const float rstd = 1.0f / sqrtf(wave_total(ss) / (float)di + p.keps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      if (c < di) st_bf4(p.key + row * di + c, x[v] * rstd * g[v]);
    }
    return;
  }
  const int qb = (int)blockIdx.x - p.key_blocks, per = (p.K + LO_Q - 1) / LO_Q, b = qb / per, k0 = (qb % per) * LO_Q;
  const int ld = NV * 256 + 4;
  {
    const int q = threadIdx.x % LO_Q, k = min(k0 + q, p.K - 1);   // (queries past the end repeat the last and are not stored)
    const long at = (long)b * di * p.K + k;
#pragma unroll 4
    for (int c = threadIdx.x / LO_Q; c < di; c += NTHREADS / LO_Q)
      tile[q * ld + c] = f_to_bf16((p.last0[at + (long)c * p.K] + p.last1[at + (long)c * p.K]) * 0.5f);
  }
  __syncthreads();
  for (int q = w; q < LO_Q && k0 + q < p.K; q += 4) {
    f4 x[NV];
    float s = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      x[v] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
      if (c < di) x[v] = ld_bf4(tile + q * ld + c);
      s += sum4(x[v]);
    }
    const float mean = wave_total(s) / (float)di;
    s = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
      if (4 * (lane + 64 * v) < di) {
        x[v] -= mean;
        s += sum4(x[v] * x[v]);
      }
    const float rstd = 1.0f / sqrtf(wave_total(s) / (float)di + p.qeps);
    uint16_t* o = p.query + ((long)b * p.K + k0 + q) * di;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      if (c < di) {
        f4 y = x[v] * rstd;
        if (p.qw) y *= ld_bf4(p.qw + c);
        if (p.qb) y += ld_bf4(p.qb + c);
        st_bf4(o + c, y);
      }
    }
  }
}

int launch_layer_out(LayerOutP& p, hipStream_t st) {
  const long key = (p.rows + 3) / 4, query = (long)p.B * ((p.K + LO_Q - 1) / LO_Q);
  if (key + query > 0x7fffffff) return (int)hipErrorInvalidValue;
  p.key_blocks = (int)key;
  const dim3 grid((unsigned)(key + query)), block(NTHREADS);
  if (p.di <= 256) hipLaunchKernelGGL(k_layer_out<1>, grid, block, 0, st, p);
  else if (p.di <= 512) hipLaunchKernelGGL(k_layer_out<2>, grid, block, 0, st, p);
  else hipLaunchKernelGGL(k_layer_out<4>, grid, block, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
