// dW = dy^T x of a decoder layer's projections (gfx950): dy (tokens, out) and x (tokens, in) bf16 row-major, dW (out, in) bf16,
// sums in fp32.  The contraction runs over the rows of both operands, and the result is only a few dozen tiles: the tokens are
// cut into `splits` parts, each wave of a workgroup takes a quarter of a part, the waves' results meet in LDS, the parts' in a
// second launch (fp32, in a fixed order).
//
// An MFMA operand holds eight consecutive rows of a column per lane: lane (i, g) loads the row pieces of its eight tokens, 4
// features of dy and 6 of x each, and eight rows' halves are paired by v_perm_b32 -- 40 of them for the 24 matrix instructions
// of a step of 32 tokens -- with no trip through LDS.  A 64 x 96 tile a wave (96 accumulators) reads 10 KB for 200 000 products.  Bound by
// the trips to memory and L2; parts are numbered so that all tiles of a part, which read the same rows, are on one XCD.
// Both launches, 8192 tokens: 288 -> 586 18.2 us, 288 -> 288 14.1 (the library's product of four slices and its sum 24.8 and
// 21.4); 2048: 11.4 and 9.7 (13.9, 13.0).  From a result of 512 x 512 on, which leaves the library's tiles no shortage of
// workgroups, that is faster (8192 tokens: 25.8 against 22.3).
// Lanes at the right edge take the last 4 (6) columns once more and store the same values as their neighbours.
#include "issm_dev.h"

namespace issm {

constexpr int DW_FA = 4, DW_FB = 6, DW_TA = 16 * DW_FA, DW_TB = 16 * DW_FB;

struct __attribute__((packed, aligned(2))) DwRowA {   // DW_FA features at any element offset
  unsigned v[DW_FA / 2];
};
struct __attribute__((packed, aligned(2))) DwRowB {
  unsigned v[DW_FB / 2];
};
// eight rows' words (two features each) -> the two features' operands
__device__ __forceinline__ void pair_rows(const unsigned (&w)[8], bf8& lo, bf8& hi) {
  uint4 a, b;
  unsigned* pa = (unsigned*)&a;
  unsigned* pb = (unsigned*)&b;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    pa[j] = __builtin_amdgcn_perm(w[2 * j + 1], w[2 * j], 0x05040100u);
    pb[j] = __builtin_amdgcn_perm(w[2 * j + 1], w[2 * j], 0x07060302u);
  }
  lo = __builtin_bit_cast(bf8, a);
  hi = __builtin_bit_cast(bf8, b);
}

__global__ __launch_bounds__(NTHREADS, 2) void k_linear_dw(LinearDwJobs jobs) {
  __shared__ f4 red[2][DW_FA * DW_FB][64];
  const bool second = (int)blockIdx.x >= jobs.blocks0;
  const LinearDwP& p = jobs.job[second ? 1 : 0];
  const int bid = (int)blockIdx.x - (second ? jobs.blocks0 : 0);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
  const int part = bid % p.splits, tile = bid / p.splits;
  const int a0 = (tile / p.btiles) * DW_TA, b0 = (tile % p.btiles) * DW_TB;
  const int ca = min(a0 + DW_FA * i, p.out - DW_FA), cb = min(b0 + DW_FB * i, p.in - DW_FB);
  const int per = p.per, t0 = min((part * 4 + w) * per, p.tokens), t1 = min(t0 + per, p.tokens);
  f4 acc[DW_FA][DW_FB];
#pragma unroll
  for (int a = 0; a < DW_FA; ++a)
#pragma unroll
    for (int b = 0; b < DW_FB; ++b) acc[a][b] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
  DwRowA ra[8];
  DwRowB rb[8];
  // a uniform base per row of the eight and one offset a lane: no address is computed per load
  const unsigned offa = 8u * g * p.out + ca, offb = 8u * g * p.in + cb;
  auto request = [&](int t) {
    const uint16_t *qa = p.dy + (long)t * p.out, *qb = p.x + (long)t * p.in;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      ra[k] = *(const DwRowA*)(qa + (long)k * p.out + offa);
      rb[k] = *(const DwRowB*)(qb + (long)k * p.in + offb);
    }
  };
  bf8 fa[DW_FA], fb[DW_FB];
  auto operands = [&](int left) {   // of the lane's eight rows, the first `left` count
#pragma unroll
    for (int c = 0; c < DW_FA / 2; ++c) {
      unsigned v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = k < left ? ra[k].v[c] : 0u;
      pair_rows(v, fa[2 * c], fa[2 * c + 1]);
    }
#pragma unroll
    for (int c = 0; c < DW_FB / 2; ++c) {
      unsigned v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = k < left ? rb[k].v[c] : 0u;
      pair_rows(v, fb[2 * c], fb[2 * c + 1]);
    }
  };
  auto products = [&]() {
#pragma unroll
    for (int a = 0; a < DW_FA; ++a)
#pragma unroll
      for (int b = 0; b < DW_FB; ++b) acc[a][b] = mfma_bf(fa[a], fb[b], acc[a][b]);
  };
  const int whole = t0 + ((t1 - t0) & ~31);
  if (t0 < whole) request(t0);
  for (int t = t0; t < whole; t += 32) {
    operands(8);
    request(min(t + 32, whole - 32));   // (the last asks for its own rows once more)
    products();
  }
  if (whole < t1) {   // fewer than 32 rows left: those behind repeat the last and count as zeros
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const long row = min(whole + 8 * g + k, t1 - 1);
      ra[k] = *(const DwRowA*)(p.dy + row * p.out + ca);
      rb[k] = *(const DwRowB*)(p.x + row * p.in + cb);
    }
    operands(t1 - whole - 8 * g);
    products();
  }
  // waves 2, 3 to waves 0, 1, then 1 to 0
#pragma unroll
  for (int half = 2; half >= 1; half >>= 1) {
    if (w >= half && w < 2 * half) {
#pragma unroll
      for (int a = 0; a < DW_FA; ++a)
#pragma unroll
        for (int b = 0; b < DW_FB; ++b) red[w - half][a * DW_FB + b][lane] = acc[a][b];
    }
    __syncthreads();
    if (w < half) {
#pragma unroll
      for (int a = 0; a < DW_FA; ++a)
#pragma unroll
        for (int b = 0; b < DW_FB; ++b) acc[a][b] += red[w][a * DW_FB + b][lane];
    }
    __syncthreads();
  }
  if (w) return;
  // accumulator r of (a, b): row a of lane 4 g + r's columns of dy, column b of the lane's of x
  float* dst = p.partial + (long)part * p.out * p.in;
#pragma unroll
  for (int a = 0; a < DW_FA; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = min(a0 + DW_FA * (4 * g + r), p.out - DW_FA) + a;
      float* q = dst + (long)o * p.in + cb;
#pragma unroll
      for (int b = 0; b < DW_FB; b += 2) {
        struct __attribute__((packed, aligned(4))) F2 { float x, y; };
        *(F2*)(q + b) = F2{acc[a][b][r], acc[a][b + 1][r]};
      }
    }
}

__global__ __launch_bounds__(NTHREADS) void k_linear_dw_sum(LinearDwJobs jobs) {
  const bool second = (int)blockIdx.x >= jobs.sums0;
  const LinearDwP& p = jobs.job[second ? 1 : 0];
  const long n = (long)p.out * p.in, e = ((long)((int)blockIdx.x - (second ? jobs.sums0 : 0)) * NTHREADS + threadIdx.x) * 2;
  if (e >= n) return;
  const bool two = e + 1 < n;
  float x = 0.0f, y = 0.0f;
#pragma unroll 8
  for (int s = 0; s < p.splits; ++s) {
    const float* q = p.partial + s * n + e;
    x += q[0];
    y += q[two ? 1 : 0];
  }
  p.dw[e] = f_to_bf16(x);
  if (two) p.dw[e + 1] = f_to_bf16(y);
}

// Parts: a workgroup a CU (two: the partial results cost more than the shorter waves save, 8192 x 288 -> 288 10.6 us -> 13.0; half of
// one: 12.6), no wave with fewer than two steps of 32 tokens, and a multiple of 8 if there are that many (a part's tiles are on one
// XCD then: 288 -> 586 in 17 parts 20.5 us, in 16 14.8).
int linear_dw_splits(long tokens, int in, int out) {
  const long tiles = (long)((out + DW_TA - 1) / DW_TA) * ((in + DW_TB - 1) / DW_TB);
  const long n = std::min(std::max(1L, 256 / std::max(1L, tiles)), std::max(1L, tokens / 256));
  return (int)(n >= 8 ? n & ~7L : n);
}

int launch_linear_dw(LinearDwJobs& j, int njobs, hipStream_t st) {
  long blocks[2] = {0, 0}, sums[2] = {0, 0};
  for (int k = 0; k < njobs; ++k) {
    LinearDwP& p = j.job[k];
    p.btiles = (p.in + DW_TB - 1) / DW_TB;
    p.per = (int)((((long)p.tokens + p.splits * 4 - 1) / (p.splits * 4) + 31) / 32 * 32);
    blocks[k] = (long)((p.out + DW_TA - 1) / DW_TA) * p.btiles * p.splits;
    sums[k] = ((long)p.out * p.in + 2 * NTHREADS - 1) / (2 * NTHREADS);
  }
  if (blocks[0] + blocks[1] > 0x7fffffff || sums[0] + sums[1] > 0x7fffffff) return (int)hipErrorInvalidValue;
  j.blocks0 = (int)blocks[0];
  j.sums0 = (int)sums[0];
  hipLaunchKernelGGL(k_linear_dw, dim3((unsigned)(blocks[0] + blocks[1])), dim3(NTHREADS), 0, st, j);
  if (hipError_t e = hipGetLastError()) return (int)e;
  hipLaunchKernelGGL(k_linear_dw_sum, dim3((unsigned)(sums[0] + sums[1])), dim3(NTHREADS), 0, st, j);
  return (int)hipGetLastError();
}

}  // namespace issm
