// A tile of a product of many tokens (linear_tile.hip), which the kernel of linear.hip that begins a layer shares.
#pragma once
#include "issm_dev.h"

namespace issm {

constexpr int LT_T = 64, LT_O = 96, LT_K = 96, LT_LD = LT_K + 8;   // tokens, outputs, contraction of a step; row stride in LDS (208 bytes: the 16
                                                                   // rows of an operand read in different banks)

struct __attribute__((packed, aligned(2))) LtPiece {   // eight values at any element offset
  unsigned v[4];
};
struct __attribute__((packed, aligned(2))) LtSix {
  unsigned v[3];
};

// NN: w is (contraction, outputs), both even; otherwise (outputs, contraction) with a contraction that is a multiple of 32.  64 rows of x and w
// are within 32-bit byte offsets (the host checks).
template <bool NN>
__device__ __forceinline__ void linear_tile(const LinearTileJob& j, int bid) {
  __shared__ __align__(16) uint16_t xs[LT_T * LT_LD], ws[LT_O * LT_LD];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
  // the last tile of either kind ends where the tensor does: what two tiles share both compute, and store the same
  const int t0 = min((bid / j.otiles) * LT_T, j.tokens - LT_T), o0 = min((bid % j.otiles) * LT_O, j.out - LT_O);
  const int in = j.in, steps = (in + LT_K - 1) / LT_K;
  constexpr int XP = LT_T * (LT_K / 8) / NTHREADS, WP = (LT_O * (LT_K / 8) + NTHREADS - 1) / NTHREADS;   // pieces a thread
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  typedef unsigned u3 __attribute__((ext_vector_type(3)));
  u4 rx[XP], rw[NN ? 1 : WP];
  u3 rn[NN ? 8 : 1];
  // the tile's rows behind buffers: what lies past the contraction's end reads zero, and no request sits behind a branch
  constexpr unsigned OUT = 0xfffffffcu;
  auto rows = [](const uint16_t* q, unsigned bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)const_cast<uint16_t*>(q), 0, bytes, 0x00027000); };
  const __amdgpu_buffer_rsrc_t bx = rows(j.x + (long)t0 * in, (unsigned)(LT_T * in) * 2u),
                               bw = NN ? rows(j.w + o0, (unsigned)((in - 1) * j.out + LT_O) * 2u) : rows(j.w + (long)o0 * in, (unsigned)(LT_O * in) * 2u);
  // eight values of a row from column k on
  auto piece = [&](const __amdgpu_buffer_rsrc_t& q, int row, int k) __attribute__((always_inline)) -> u4 {
    return __builtin_amdgcn_raw_buffer_load_b128(q, k < in ? (unsigned)(row * in + k) * 2u : OUT, 0, 0);
  };
  auto request = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < XP; ++q) {
      const int e = tid + q * NTHREADS;
      rx[q] = piece(bx, e / (LT_K / 8), k0 + e % (LT_K / 8) * 8);
    }
    if constexpr (!NN) {
#pragma unroll
      for (int q = 0; q < WP; ++q) {
        const int e = min(tid + q * NTHREADS, LT_O * (LT_K / 8) - 1);
        rw[q] = piece(bw, e / (LT_K / 8), k0 + e % (LT_K / 8) * 8);
      }
    } else {
      const int n0 = k0 + 8 * min(tid >> 4, LT_K / 8 - 1);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        rn[k] = __builtin_amdgcn_raw_buffer_load_b96(bw, n0 + k < in ? (unsigned)((n0 + k) * j.out + 6 * (tid & 15)) * 2u : OUT, 0, 0);
    }
  };
  auto keep = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < XP; ++q) {
      const int e = tid + q * NTHREADS;
      u4 v = rx[q];
      if constexpr (NN) {   // (a piece across the end of its row goes on in the next)
        const int left = in - (k0 + e % (LT_K / 8) * 8);
#pragma unroll
        for (int d = 0; d < 4; ++d) v[d] = left > 2 * d ? v[d] : 0u;
      }
      *(u4*)(xs + e / (LT_K / 8) * LT_LD + e % (LT_K / 8) * 8) = v;
    }
    if constexpr (!NN) {
#pragma unroll
      for (int q = 0; q < WP; ++q) {
        const int e = tid + q * NTHREADS;
        if (e < LT_O * (LT_K / 8)) *(u4*)(ws + e / (LT_K / 8) * LT_LD + e % (LT_K / 8) * 8) = rw[q];
      }
    } else if (tid < 16 * (LT_K / 8)) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        u4 lo, hi;   // columns 2 c, 2 c + 1 of eight rows
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          lo[k] = __builtin_amdgcn_perm(rn[2 * k + 1][c], rn[2 * k][c], 0x05040100u);
          hi[k] = __builtin_amdgcn_perm(rn[2 * k + 1][c], rn[2 * k][c], 0x07060302u);
        }
        uint16_t* d = ws + (6 * (tid & 15) + 2 * c) * LT_LD + 8 * (tid >> 4);
        *(u4*)d = lo;
        *(u4*)(d + LT_LD) = hi;
      }
    }
  };
  // wave (wm, wn): two blocks of 16 tokens, three of 16 outputs, five operands read for six products (one by six: seven)
  const int wm = w & 1, wn = w >> 1;
  f4 acc[2][3];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int f = 0; f < 3; ++f) acc[m][f] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
  const uint16_t *qx = xs + (wm * 32 + i) * LT_LD + 8 * g, *qw = ws + (wn * 48 + i) * LT_LD + 8 * g;
  request(0);
  for (int s = 0; s < steps; ++s) {
    if (s) __syncthreads();   // the step before has been read
    keep(s * LT_K);
    __syncthreads();
    if (s + 1 < steps) request((s + 1) * LT_K);
#pragma unroll
    for (int u = 0; u < LT_K / 32; ++u)
      if (s * LT_K + 32 * u < in) {   // uniform
        bf8 fx[2], fw[3];
#pragma unroll
        for (int m = 0; m < 2; ++m) fx[m] = *(const bf8*)(qx + 16 * m * LT_LD + 32 * u);
#pragma unroll
        for (int f = 0; f < 3; ++f) fw[f] = *(const bf8*)(qw + 16 * f * LT_LD + 32 * u);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int f = 0; f < 3; ++f) acc[m][f] = mfma_bf(fw[f], fx[m], acc[m][f]);
      }
  }
  __syncthreads();
  // accumulator r of (m, f): output 16 f + 4 g + r of token 16 m + i of the wave's (LDS instructions of a wave are carried out in order)
  uint16_t* own = xs + wm * 32 * LT_LD + wn * 48;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int f = 0; f < 3; ++f) *(bf4*)(own + (16 * m + i) * LT_LD + 16 * f + 4 * g) = __builtin_convertvector(acc[m][f], bf4);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int e = lane + 64 * q, row = e / 6, c = e % 6 * 8;
    const u4 v = *(const u4*)(own + row * LT_LD + c);
    *(LtPiece*)(j.y + (long)(t0 + wm * 32 + row) * j.out + o0 + wn * 48 + c) = LtPiece{{v[0], v[1], v[2], v[3]}};
  }
}

}  // namespace issm
