// Queries <-> initial / final states: the two rearrangements around the scan in MultiHeadISSMScan.forward,
//   initial_states = rearrange(query_proj(in_query), "b l (h hd) -> b h hd l")        (models/dest_module.py:537-538)
//   last_states    = rearrange((last_states + last_states_back) / 2, "b h p l -> b l (h p)")   (:575, :582)
// and their gradients, as one batched transpose with the average and the dtype conversion folded in (gfx950):
//   out[b][c][r] = alpha * (in0[b][r][c] + in1[b][r][c])        in (B, R, C), out (B, C, R), in1 optional.
// As tensor ops each is a strided copy (uncoalesced on one side) plus separate add / scale / cast kernels; here a
// 64 x 64 tile goes through LDS so that both sides move 64 consecutive elements per wave row.
#include "transpose_dev.h"

namespace issm {

template <bool IN_BF, bool OUT_BF>
__global__ __launch_bounds__(NTHREADS) void k_transpose_states(TrP p) {
  __shared__ float tile[64][65];
  transpose_tile<IN_BF, OUT_BF>(p, blockIdx.x * 64, blockIdx.y * 64, blockIdx.z, tile);
}

// The gradients of a layer's small parameters from what the backwards left of them (issm_layer_grads), and the queries' gradient turned, in
// one launch.  A few thousand results from 10 MB at most: each kind's workgroups are a few round trips to memory, and together they take the time of
// the longest: 8.7 us at 8 x 1024 tokens, 288 features and 256 queries, where the three sums (5.3, 7.1 and 7.4 us), A_log's sum and product, the
// concatenation, the conversion and the transposition were eight launches and 43 us.
//
// Column `col` of src (rows, ncol), summed by NTHREADS / COLS threads that take every NTHREADS / COLS-th row; the sum in those of row 0.  The
// adds are a chain in a fixed order, but the loads of eight rounds travel together.
template <int COLS>
__device__ __forceinline__ float column_sum(const float* src, int rows, int ncol, int col, float* red) {
  constexpr int G = NTHREADS / COLS;
  const int g = threadIdx.x / COLS;
  float a0 = 0.0f, a1 = 0.0f;
  if (col < ncol) {
    int r = g;
#pragma unroll 8
    for (; r + G < rows; r += 2 * G) {
      a0 += src[(long)r * ncol + col];
      a1 += src[(long)(r + G) * ncol + col];
    }
    if (r < rows) a0 += src[(long)r * ncol + col];
  }
  red[threadIdx.x] = a0 + a1;
  __syncthreads();
  float t = 0.0f;
  if (g == 0)
#pragma unroll
    for (int k = 0; k < G; ++k) t += red[k * COLS + threadIdx.x];
  return t;
}

template <bool OUT_BF>
__global__ __launch_bounds__(NTHREADS) void k_layer_grads(LayerGradsP p, TrP t) {
  __shared__ float tile[64][65];
  float* const red = &tile[0][0];
  const int b = blockIdx.x, lane = threadIdx.x & 63;
  if (b >= p.b_tr) return transpose_nth<false, OUT_BF>(t, b - p.b_tr, tile);
  const int conv = 16 * p.C, gen = 16 * p.R0;   // results of the convolutions and of the generation
  auto put = [&](int e, float v) { stv(p.out, e, p.bf16, v); };
  if (b < p.b_gen) {
    const int col = b * 16 + (threadIdx.x & 15), c = col % p.C, sj = col / p.C, j = sj & 7;
    const float v = column_sum<16>(p.conv, p.conv_rows, conv, col, red);
    if (threadIdx.x < 16) put((sj >> 3) * 8 * p.C + (j < 7 ? c * 7 + j : 7 * p.C + c), v);
  } else if (b < p.b_bias) {
    const int col = (b - p.b_gen) * 8 + (threadIdx.x & 7);
    const float v = column_sum<8>(p.gen, p.gen_rows, gen, col, red);
    if (threadIdx.x < 8) put(conv + col, v);
  } else if (b < p.b_norm) {
    const int col = (b - p.b_bias) * 8 + (threadIdx.x & 7);
    const float v = column_sum<8>(p.gen_bias, p.gen_rows, p.R0, col, red);
    if (threadIdx.x < 8 && col < p.H) put(conv + gen + col, v);
  } else if (b < p.b_A) {
    const int col = (b - p.b_norm) * 8 + (threadIdx.x & 7);
    const float v = column_sum<8>(p.norm, p.norm_rows, p.di, col, red);
    if (threadIdx.x < 8 && col < p.di) put(conv + gen + 2 * p.H + p.nD + col, v);
  } else if (b < p.b_D) {
    const int h = (b - p.b_A) * 4 + (threadIdx.x >> 6);
    if (h >= p.H) return;
    float v = 0.0f;
#pragma unroll 4
    for (int k = lane; k < p.K; k += 64) v += p.dA[(long)h * p.K + k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) put(conv + gen + p.H + h, p.K ? v * p.A[(long)h * p.K] : 0.0f);
  } else {
    const int e = (b - p.b_D) * NTHREADS + threadIdx.x;
    if (e < p.nD) put(conv + gen + 2 * p.H + e, p.dD[e]);
  }
}

int launch_layer_grads(LayerGradsP& p, const TrP& t, hipStream_t st) {
  p.b_gen = p.C;   // 16 C columns, 16 a workgroup
  p.b_bias = p.b_gen + 2 * p.R0;
  p.b_norm = p.b_bias + (p.H + 7) / 8;
  p.b_A = p.b_norm + (p.di + 7) / 8;
  p.b_D = p.b_A + (p.H + 3) / 4;
  p.b_tr = p.b_D + (p.nD + NTHREADS - 1) / NTHREADS;
  const long blocks = p.b_tr + transpose_tiles(t);
  if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
  if (t.out_dt) hipLaunchKernelGGL(k_layer_grads<true>, dim3((unsigned)blocks), dim3(NTHREADS), 0, st, p, t);
  else hipLaunchKernelGGL(k_layer_grads<false>, dim3((unsigned)blocks), dim3(NTHREADS), 0, st, p, t);
  return (int)hipGetLastError();
}

int launch_transpose_states(const TrP& p, hipStream_t st) {
  const dim3 g((p.C + 63) / 64, (p.R + 63) / 64, p.B), b(NTHREADS);
  if (p.in_dt) {
    if (p.out_dt) hipLaunchKernelGGL((k_transpose_states<true, true>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_transpose_states<true, false>), g, b, 0, st, p);
  } else {
    if (p.out_dt) hipLaunchKernelGGL((k_transpose_states<false, true>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_transpose_states<false, false>), g, b, 0, st, p);
  }
  return (int)hipGetLastError();
}

}  // namespace issm
