// What lies behind a decoder layer's scan where no gradient is asked for (gfx950), bf16:
//   key    = RMSNorm(bf16(y0 + y1) * silu(z)) * w          a wave a row of the (batch x seqlen, d_inner) scan outputs
//   query  = LayerNorm(bf16((last0 + last1) / 2)^T)         the d_inner values of a few queries, fp32 and one per state row, meet in LDS as
//                                                           bf16 (issm_transpose_states' result)
// and their output projections: k_layer_end, which is what the layer takes, and k_layer_out, the same without the projections, for
// callers that have something else behind the norms.  Each line was a launch or two of its own (add, norm, transpose, LayerNorm), 3 to
// 4 us whatever its size and as much again to issue; at one scene (1024 tokens, 256 queries, 288 features) the four took 15 us, k_layer_out 6.
// Bound by the launch and one trip to memory.  The sums and averages are rounded to bf16 as the separate kernels stored them.
#include <algorithm>

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

// The gated norm of row `row`, by a wave: four features a lane and vector.
template <int NV>
__device__ __forceinline__ void key_norm(const LayerOutP& p, long row, int lane, uint16_t* to) {
  const int di = p.di;
  f4 x[NV], z[NV], kw[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = min(4 * (lane + 64 * v), di - 4);   // (past the end: the last vector again, not counted)
    x[v] = ld_bf4(p.y0 + row * di + c) + ld_bf4(p.y1 + row * di + c);
    z[v] = ld_bf4(p.z + row * p.zs + c);
    kw[v] = ld_bf4(p.kw + c);
  }
  float ss = 0.0f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    x[v] = round_bf4(x[v]);
#pragma unroll
    for (int r = 0; r < 4; ++r) x[v][r] *= z[v][r] * sigmoidf_(z[v][r]);
    if (4 * (lane + 64 * v) < di) ss += sum4(x[v] * x[v]);
  }
  const float rstd = 1.0f / sqrtf(wave_total(ss) / (float)di + p.keps);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = 4 * (lane + 64 * v);
    if (c < di) st_bf4(to + c, x[v] * rstd * kw[v]);
  }
}

// The LayerNorm of a query whose values lie in LDS, by a wave.
template <int NV>
struct QueryNorm {
  f4 w[NV], b[NV];
  __device__ __forceinline__ QueryNorm(const LayerOutP& p, int lane) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = min(4 * (lane + 64 * v), p.di - 4);
      w[v] = (f4){1.0f, 1.0f, 1.0f, 1.0f};
      b[v] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
      if (p.qw) w[v] = ld_bf4(p.qw + c);   // uniform
      if (p.qb) b[v] = ld_bf4(p.qb + c);
    }
  }
  __device__ __forceinline__ void operator()(const LayerOutP& p, int lane, const uint16_t* from, uint16_t* to) const {
    const int di = p.di;
    f4 x[NV];
    float s = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      x[v] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
      if (c < di) x[v] = ld_bf4(from + c);
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
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int c = 4 * (lane + 64 * v);
      if (c < di) st_bf4(to + c, x[v] * rstd * w[v] + b[v]);
    }
  }
};

constexpr int LO_Q = 8;   // queries a workgroup: 32-byte pieces of a state row and still 32 workgroups at one scene

template <int NV>
__global__ __launch_bounds__(NTHREADS) void k_layer_out(LayerOutP p) {
  __shared__ uint16_t tile[LO_Q * (NV * 256 + 4)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, di = p.di;
  if ((int)blockIdx.x < p.key_blocks) {
    const long row = (long)blockIdx.x * 4 + w;
    if (row < p.rows) key_norm<NV>(p, row, lane, p.key + row * di);
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
  const QueryNorm<NV> norm(p, lane);
  __syncthreads();
  for (int q = w; q < LO_Q && k0 + q < p.K; q += 4) norm(p, lane, tile + q * ld, p.query + ((long)b * p.K + k0 + q) * di);
}

// The norms and the output projections, one launch: a workgroup of sixteen waves takes 16 rows (or queries) through the
// norm into LDS, a wave a row, and multiplies them with the weights of up to 256 outputs, 16 a wave, whose fragments it has asked for
// before the rows.  The two launches took 6.0 and 5.1 us at one scene, each a trip to memory and a little arithmetic.  A few hundred
// instructions a wave decide here: with four waves a workgroup and four rows a wave it took 10.2 us.  (The norm of a row is
// computed once for each workgroup that shares its outputs.)  NC: 64 features each; N: fragments in flight.
template <int NC, int N>
__global__ __launch_bounds__(1024) void k_layer_end(LayerOutP p, LinearP q, int per_block0, int per_block1) {
  warm_first<sizeof(LayerOutP) + sizeof(LinearP) + 8>();
  constexpr int NV = (NC + 3) / 4, LD = NC * 64 + 8;
  __shared__ __align__(16) uint16_t tile[16 * LD];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4, di = p.di;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool second = (int)blockIdx.x >= p.key_blocks;
  const int out = second ? q.job[1].out : q.job[0].out, nblk = second ? q.job[1].oblocks : q.job[0].oblocks;
  const int per = second ? per_block1 : per_block0, steps = di / 32;   // per: 16 outputs each, of a workgroup
  const uint16_t* wt = second ? q.job[1].w : q.job[0].w;
  const int bid = (int)blockIdx.x - (second ? p.key_blocks : 0), tb = bid / nblk, o0 = ((bid % nblk) * per + w) * 16;
  const bool mine = w < per && o0 < out;   // uniform
  const bf8* wa = (const bf8*)(wt + (long)min(o0 + i, out - 1) * di) + g;
  bf8 fa[N];
  auto request = [&](int s0) {
#pragma unroll
    for (int u = 0; u < N; ++u) fa[u] = wa[4 * min(s0 + u, steps - 1)];
  };
  request(0);
  uint16_t* row_of = tile + w * LD;
  long out_row, rows_left;   // the workgroup's first row of the product, how many of its 16 exist
  if (!second) {
    out_row = (long)tb * 16;
    rows_left = p.rows - out_row;
    key_norm<NV>(p, min(out_row + w, p.rows - 1), lane, row_of);
  } else {
    const int perb = (p.K + 15) / 16, b = tb / perb, k0 = (tb % perb) * 16;
    out_row = (long)b * p.K + k0;
    rows_left = p.K - k0;
    {
      const int qi = threadIdx.x & 15, c0 = threadIdx.x >> 4;
      const long at = (long)b * di * p.K + min(k0 + qi, p.K - 1);   // (queries past the end repeat the last and are not stored)
      float a0[NC], a1[NC];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        const long o = at + (long)min(c0 + 64 * m, di - 1) * p.K;
        a0[m] = p.last0[o];
        a1[m] = p.last1[o];
      }
#pragma unroll
      for (int m = 0; m < NC; ++m)
        if (c0 + 64 * m < di) tile[qi * LD + c0 + 64 * m] = f_to_bf16((a0[m] + a1[m]) * 0.5f);
    }
    const QueryNorm<NV> norm(p, lane);
    __syncthreads();
    norm(p, lane, row_of, row_of);
  }
  __syncthreads();
  if (!mine) return;
  f4 y4 = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < steps; s0 += N) {
    if (s0) request(s0);
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (s0 + u < steps) y4 = mfma_bf(fa[u], *(const bf8*)(tile + i * LD + 32 * (s0 + u) + 8 * g), y4);   // uniform
  }
  if (i >= rows_left) return;
  const int o = o0 + 4 * g;
  uint16_t* y = (second ? q.job[1].y : q.job[0].y) + (out_row + i) * out + o;
  if (o + 4 <= out) {
    st_bf4(y, y4);
  } else {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (o + r < out) y[r] = f_to_bf16(y4[r]);
  }
}

int launch_layer_end(LayerOutP& p, LinearP& q, hipStream_t st) {
  const long tiles[2] = {(p.rows + 15) / 16, (long)p.B * ((p.K + 15) / 16)}, all = tiles[0] + tiles[1];
  long blocks[2];
  int per[2];
  for (int k = 0; k < 2; ++k) {
    // the outputs of a tile of rows shared by as many workgroups as give no CU a second one, 16 outputs a wave
    const int groups = (q.job[k].out + 15) / 16, least = (groups + 15) / 16;
    const int want = std::max(least, (int)std::min((long)groups, all ? NCU / all : 1));
    per[k] = want ? (groups + want - 1) / want : 1;
    q.job[k].oblocks = (groups + per[k] - 1) / per[k];
    blocks[k] = tiles[k] * q.job[k].oblocks;
  }
  if (blocks[0] + blocks[1] > 0x7fffffff) return (int)hipErrorInvalidValue;
  if (blocks[0] + blocks[1] == 0) return 0;
  p.key_blocks = (int)blocks[0];
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)(blocks[0] + blocks[1])), dim3(1024), 0, st, p, q, per[0], per[1]); };
  // (fragments in flight: all there are, up to 320 features; 320, four scenes of 1024 tokens, a layer 172 us with eight of ten, 168 so)
  if (p.di <= 256) go(&k_layer_end<4, 8>);
  else if (p.di <= 320) go(&k_layer_end<5, 10>);
  else if (p.di <= 512) go(&k_layer_end<8, 8>);
  else go(&k_layer_end<16, 4>);
  return (int)hipGetLastError();
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
