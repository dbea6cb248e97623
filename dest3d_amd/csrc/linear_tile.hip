// y = x W^T and dx = dy W of a decoder layer's projections where thousands of tokens meet a few hundred features (gfx950), bf16 operands,
// fp32 accumulation.  Up to two such products share a launch.
//
// At these sizes a product is a few memory trips long whoever computes it (8192 x 288 -> 288: 1.4 GFLOP and 9.6 MB, 2 us of either), and its
// time is those trips and how many of them the chip has under way.  Workgroup = 64 tokens x 96 outputs, four waves of 32 x 48: enough
// workgroups that every CU has one or two to run beside another.  The contraction goes through LDS 96 at a time, the next 96 requested in pieces
// of rows while these are multiplied (pieces of 64 bytes in the layout of the matrix operands, as linear.hip has them, are 64 look-ups in
// the L1 a load).  dx contracts over W's rows: a thread takes eight rows of six columns, whose halves v_perm_b32 pairs into the operand's
// order.  Results leave through the LDS that held the wave's tokens, in pieces of rows again.
// us, with the library's product in brackets: y, 288 -> 586, 2048, 8192 and 32768 tokens 5.0 (6.7), 10.6 (13.0), 34.7 (38.4), 288 -> 288 4.5 (5.4), 6.2
// (8.9), 14.9 (21.6); dx, 586 -> 288, 8.5 (9.2), 11.6 (16.3), 29.5 (37.8), 288 -> 288 5.1 (6.2), 6.8 (10.4), 16.0 (22.3).  (A wave of 16 tokens and all 96
// outputs reads seven operands for six products where this takes five: 8192 x 288 -> 586 11.9.)
#include "linear_tile_dev.h"

namespace issm {

template <bool NN>
__global__ __launch_bounds__(NTHREADS) void k_linear_tile(LinearTileP p) {
  const int wg = xcd_remap(blockIdx.x, gridDim.x);   // (an XCD's workgroups read the same tokens)
  const bool second = wg >= p.blocks0;
  linear_tile<NN>(p.job[second ? 1 : 0], wg - (second ? p.blocks0 : 0));
}

bool linear_tile_takes(long tokens, int in, int out, bool nn) {
  return tokens >= LT_T && out >= LT_O && (nn ? in >= 2 && !((in | out) & 1) : in >= 32 && in % 32 == 0) && (long)in * out < (1L << 30) && in < (1 << 22);
}

int launch_linear_tile(LinearTileP& p, int njobs, bool nn, hipStream_t st) {
  long blocks[2] = {0, 0};
  for (int k = 0; k < njobs; ++k) {
    p.job[k].otiles = (p.job[k].out + LT_O - 1) / LT_O;
    blocks[k] = (long)((p.job[k].tokens + LT_T - 1) / LT_T) * p.job[k].otiles;
  }
  if (blocks[0] + blocks[1] > 0x7fffffff) return (int)hipErrorInvalidValue;
  p.blocks0 = (int)blocks[0];
  const dim3 grid((unsigned)(blocks[0] + blocks[1])), block(NTHREADS);
  if (nn) hipLaunchKernelGGL(k_linear_tile<true>, grid, block, 0, st, p);
  else hipLaunchKernelGGL(k_linear_tile<false>, grid, block, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
