// y = x W^T of a decoder layer's projections where a scene or two of tokens meet a few hundred features (gfx950), bf16 operands,
// fp32 accumulation: x (tokens, in), W (out, in), y (tokens, out).  Up to two such products share a launch.
//
// At these sizes a product is a few microseconds whoever computes it, and what counts is what it costs to launch: a library
// product takes 19 us of host time to issue, 4.6 here; a decoder layer has four, and six layers on one scene (1024 tokens, 256
// queries) ran at the pace of the host: 1180 - 1350 us from process to process, 885 with this.  Without a gradient a layer's first
// two are one such launch, the queries turned into the layout of the scan's states on the way (the last two: layer_out.hip).  Both operands have the contraction index contiguous, which is the operand layout of
// v_mfma_f32_16x16x32_bf16 as it lies in memory: a wave asks for all fragments of its 16 tokens and 32 outputs at once (27 loads
// of 16 bytes a lane at 288 features) and multiplies as they arrive; there is nothing to share through LDS that L1 does not
// share.  1024 x 288 -> 586: 6.3 us (library 6.1), 288: 4.5 (5.1).  With more tokens the fragments' 64-byte pieces
// of 16 rows a load are what it pays for, and staging tiles through LDS wins (linear_tile.hip): 8192 x 288 -> 586 21 us, in tiles 10.6.
#include "layer_params.h"
#include "linear_tile_dev.h"

namespace issm {

struct __attribute__((packed, aligned(2))) LinearOut {   // four outputs; rows of an odd number of them promise no alignment
  bf4 v;
};

// N: fragments in flight.  TURN: the product is stored transposed within each j.turn tokens (queries as the scan's initial
// states); the operands change places, and a lane holds four tokens of an output instead of four outputs of a token.
template <int N, bool TURN>
__device__ __forceinline__ void linear_block(const LinearJob& j, int bid) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int t = (bid / j.oblocks) * 64 + (threadIdx.x >> 6) * 16 + i, o0 = (bid % j.oblocks) * 32;
  const long in = 32L * j.steps;
  const bf8* x = (const bf8*)(j.x + (long)min(t, j.tokens - 1) * in) + g;
  const bf8 *wa = (const bf8*)(j.w + (long)min(o0 + i, j.out - 1) * in) + g,
            *wb = (const bf8*)(j.w + (long)min(o0 + 16 + i, j.out - 1) * in) + g;
  f4 ya = {0, 0, 0, 0}, yb = {0, 0, 0, 0};
  for (int s0 = 0; s0 < j.steps; s0 += N) {
    bf8 fx[N], fa[N], fb[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int s = 4 * min(s0 + u, j.steps - 1);
      fx[u] = x[s];
      fa[u] = wa[s];
      fb[u] = wb[s];
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (s0 + u < j.steps) {   // uniform
        ya = TURN ? mfma_bf(fx[u], fa[u], ya) : mfma_bf(fa[u], fx[u], ya);
        yb = TURN ? mfma_bf(fx[u], fb[u], yb) : mfma_bf(fb[u], fx[u], yb);
      }
  }
  if constexpr (TURN) {
    const int t4 = t - i + 4 * g, row = t4 / j.turn, col = t4 % j.turn;
    auto put = [&](int o, f4 v) {
      if (o >= j.out) return;
      uint16_t* y = j.y + ((long)row * j.out + o) * j.turn + col;
      if (col + 4 <= j.turn && t4 + 4 <= j.tokens) {
        ((LinearOut*)y)->v = __builtin_convertvector(v, bf4);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t4 + r < j.tokens) j.y[((long)((t4 + r) / j.turn) * j.out + o) * j.turn + (t4 + r) % j.turn] = f_to_bf16(v[r]);
      }
    };
    put(o0 + i, ya);
    put(o0 + 16 + i, yb);
    return;
  }
  if (t >= j.tokens) return;
  uint16_t* y = j.y + (long)t * j.out;
  auto put = [&](int o, f4 v) {
    if (o + 4 <= j.out) {
      ((LinearOut*)(y + o))->v = __builtin_convertvector(v, bf4);
    } else {
#pragma unroll
      for (int r = 0; r < 3; ++r)
        if (o + r < j.out) y[o + r] = f_to_bf16(v[r]);
    }
  };
  put(o0 + 4 * g, ya);
  put(o0 + 16 + 4 * g, yb);
}

template <int N>
__global__ __launch_bounds__(NTHREADS) void k_linear(LinearP p) {
  const bool second = (int)blockIdx.x >= p.blocks0;
  const LinearJob& j = p.job[second ? 1 : 0];
  const int bid = (int)blockIdx.x - (second ? p.blocks0 : 0);
  if (j.turn) linear_block<N, true>(j, bid);
  else linear_block<N, false>(j, bid);
}

// The products and, in the blocks behind theirs, the layer's small parameters (issm_layer_in): 7.6 us where the two launches
// took 6.8 and 3.1.
// (Compiled without -ffast-math for its exp.)
template <int N>
__global__ __launch_bounds__(NTHREADS) void k_layer_in(LinearP p, LayerParamsP q) {
  warm_first<sizeof(LinearP) + sizeof(LayerParamsP)>();
  if ((int)blockIdx.x >= p.blocks1) return layer_params_entry(q, ((int)blockIdx.x - p.blocks1) * NTHREADS + threadIdx.x);
  const bool second = (int)blockIdx.x >= p.blocks0;
  const LinearJob& j = p.job[second ? 1 : 0];
  const int bid = (int)blockIdx.x - (second ? p.blocks0 : 0);
  if (j.turn) linear_block<N, true>(j, bid);
  else linear_block<N, false>(j, bid);
}

// The same with the first product in tiles, where issm_linear_fwd takes them, and, without parameters, a pair of which one product alone is (8192 x 288 ->
// 586 beside 32 x 288 -> 288 20.7 -> 10.2 us).  A layer without a gradient, us, scenes of 1024 tokens and 256
// queries: 288 features, 1, 4 and 8 scenes 58.2 -> 57.8, 135 -> 129, 232 -> 223; 96, 16: 293 -> 288; 320, 3: 131 -> 113; 512, 2: 126 -> 107.
template <int N>
__global__ __launch_bounds__(NTHREADS) void k_layer_in_tile(LinearTileP t, LinearP p, LayerParamsP q) {
  warm_first<sizeof(LinearTileP) + sizeof(LinearP) + sizeof(LayerParamsP)>();
  const int wg = blockIdx.x;
  if (wg >= p.blocks1) return layer_params_entry(q, (wg - p.blocks1) * NTHREADS + threadIdx.x);
  if (wg < t.blocks0) return linear_tile<false>(t.job[0], xcd_remap(wg, t.blocks0));
  const LinearJob& j = p.job[1];
  if (j.turn) linear_block<N, true>(j, wg - t.blocks0);
  else linear_block<N, false>(j, wg - t.blocks0);
}

int launch_layer_in_tile(LinearTileP& t, LinearP& p, const LayerParamsP& q, hipStream_t st) {
  t.job[0].otiles = (t.job[0].out + LT_O - 1) / LT_O;
  p.job[1].oblocks = (p.job[1].out + 31) / 32;
  const long tiles = (long)((t.job[0].tokens + LT_T - 1) / LT_T) * t.job[0].otiles,
             blocks = tiles + (long)((p.job[1].tokens + 63) / 64) * p.job[1].oblocks, params = ((long)q.total + q.H * q.K + NTHREADS - 1) / NTHREADS;
  if (blocks + params > 0x7fffffff) return (int)hipErrorInvalidValue;
  t.blocks0 = (int)tiles;
  p.blocks1 = (int)blocks;
  const dim3 grid((unsigned)(blocks + params)), block(NTHREADS);
  if (p.job[1].steps % 9 == 0) hipLaunchKernelGGL(k_layer_in_tile<9>, grid, block, 0, st, t, p, q);
  else hipLaunchKernelGGL(k_layer_in_tile<8>, grid, block, 0, st, t, p, q);
  return (int)hipGetLastError();
}

int launch_linear(LinearP& p, int njobs, const LayerParamsP* q, hipStream_t st) {
  long blocks[2] = {0, 0};
  for (int k = 0; k < njobs; ++k) {
    p.job[k].oblocks = (p.job[k].out + 31) / 32;
    blocks[k] = (long)((p.job[k].tokens + 63) / 64) * p.job[k].oblocks;
  }
  const long params = q ? ((long)q->total + q->H * q->K + NTHREADS - 1) / NTHREADS : 0;
  if (blocks[0] + blocks[1] + params > 0x7fffffff) return (int)hipErrorInvalidValue;
  p.blocks0 = (int)blocks[0];
  p.blocks1 = (int)(blocks[0] + blocks[1]);
  const dim3 grid((unsigned)(blocks[0] + blocks[1] + params)), block(NTHREADS);
  if (q) {
    if (p.job[0].steps % 9 == 0) hipLaunchKernelGGL(k_layer_in<9>, grid, block, 0, st, p, *q);
    else hipLaunchKernelGGL(k_layer_in<8>, grid, block, 0, st, p, *q);
    return (int)hipGetLastError();
  }
  // nine fragments where they come out even (288 features), eight otherwise
  if (p.job[0].steps % 9 == 0) hipLaunchKernelGGL(k_linear<9>, grid, block, 0, st, p);
  else hipLaunchKernelGGL(k_linear<8>, grid, block, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
