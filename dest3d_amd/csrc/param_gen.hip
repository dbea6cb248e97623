// Generation of the scan's dt / B / C from the pairwise distance encoding (gfx950).
//
// DEST builds the per-(token, query) scan parameters as tiny projections of `dist` (tokens, K, M):
//   base[r][k] = sum_m W[r][m] dist[k][m],   r = 0 .. R0-1,  R0 = H + 2G  (dt heads, B groups, C groups)
//   dt[h][k] = base[h][k] + bias[h],  B[g][k] = base[H+g][k] + bias[H+g],  C[g][k] = base[H+G+g][k] + bias[H+G+g]
// and, for the reversed-order scan, a second B / C pair from the same base rows with their own biases
// (models/dest_module.py:543-553).  As library GEMMs these are thousands of (R0 x M)(M x K) products with
// M = 16: launch- and layout-bound.  Here one pass reads `dist` once and writes every output; the backward is
// one pass as well (ddist, per-token bias gradients, per-workgroup partials of dW) plus a fixed-order
// reduction of the partials.  Everything is memory bound; arithmetic is fp32.
#include "dwconv_dev.h"

namespace issm {

constexpr int PG_MAXR0 = 12;  // largest H + 2G built (three 4-row steps of the matrix instruction)
constexpr int PG_M = 16;      // distance encoding width this kernel is built for
constexpr int PG_TOK = 4;     // tokens per workgroup in the backward (one per wave)
constexpr int PG_LDR = 144;    // bytes of a staged gradient row: 128, and 16 so that the 16 rows' pieces of 8 lie in different banks
constexpr int PG_LDT = 20;    // row stride of the backward's 16 x 16 LDS tiles (column-wise reads of four row groups
                              // fall into different banks; rows stay 8- and 16-byte aligned)

// sum over the 16 lanes that share lane >> 4; valid in the lane with (lane & 15) == 15
__device__ __forceinline__ float row_sum16_(float v) {
#define ISSM_PG_DPP_ADD(ctrl) \
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true))
  ISSM_PG_DPP_ADD(0x111);  // row_shr:1
  ISSM_PG_DPP_ADD(0x112);  // row_shr:2
  ISSM_PG_DPP_ADD(0x114);  // row_shr:4
  ISSM_PG_DPP_ADD(0x118);  // row_shr:8
#undef ISSM_PG_DPP_ADD
  return v;
}

template <bool BF>
__device__ __forceinline__ void load_row16(const void* p, long off, float (&v)[PG_M]) {
  if (BF) {
    const uint4* q = (const uint4*)((const uint16_t*)p + off);
    const uint4 a = q[0], b = q[1];
    const unsigned w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  } else {
    const f4* q = (const f4*)((const float*)p + off);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f4 a = q[i];
      v[4 * i] = a.x; v[4 * i + 1] = a.y; v[4 * i + 2] = a.z; v[4 * i + 3] = a.w;
    }
  }
}
template <bool BF>
__device__ __forceinline__ void store_row16(void* p, long off, const float (&v)[PG_M]) {
  if (BF) {
    unsigned w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = (unsigned)f_to_bf16(v[2 * i]) | ((unsigned)f_to_bf16(v[2 * i + 1]) << 16);
    uint4* q = (uint4*)((uint16_t*)p + off);
    q[0] = make_uint4(w[0], w[1], w[2], w[3]);
    q[1] = make_uint4(w[4], w[5], w[6], w[7]);
  } else {
    f4* q = (f4*)((float*)p + off);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = (f4){v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
  }
}
template <bool BF>
__device__ __forceinline__ float ld1(const void* p, long i) {
  return BF ? bf16_to_f(((const uint16_t*)p)[i]) : ((const float*)p)[i];
}
template <bool BF>
__device__ __forceinline__ void st1(void* p, long i, float v) {
  if (BF) ((uint16_t*)p)[i] = f_to_bf16(v); else ((float*)p)[i] = v;
}

// Forward: thread = (token, KV adjacent k) -- KV = 2 whenever K is even, so that every store instruction of a wave
// covers 256 (bf16) or 512 bytes instead of 128 / 256.  W and the token's biases are uniform across the lanes of a
// token: scalar operands.
// TOK: the biases come from the tensors their producers wrote (the projection's row, the convolution's tail) instead of a
// gathered fp32 copy, which cost two launches and a pass of its own.  The workgroup's tokens (two at 256 queries) are gathered
// into LDS, a value per thread; each lane loading its own row in 2-byte pieces took 55 us at 8192 tokens x 256, this 36,
// reading the gathered copy 35.
// RAW: dt before softplus and weight is kept for the backward where there are weights (a scene of 1024 tokens x 256: 10.4 us,
// 9.5 without).
// CONV: B and C's biases are the convolutions' outputs for the last 2G channels, computed here from their inputs.
// FAR: two tokens' rows are not within 31-bit byte offsets (KV = 1).
template <bool BF, int KV, bool TOK, bool RAW, bool CONV, bool FAR>
__device__ __forceinline__ void pgen_fwd(const PGenP& p, const DwConvP& conv, int block) {
  const int R0 = p.H + 2 * p.G, R = R0 + (p.has_back ? 2 * p.G : 0);
  const int per_tok = (p.K + KV - 1) / KV;  // threads per token
  extern __shared__ float tok_bias[];   // TOK: (tokens of the workgroup, R), rows as in p.bias
  // the workgroup's first token (uniform), the thread's place from it on
  const long t0 = (long)block * NTHREADS / per_tok;
  const unsigned skipped = (unsigned)((long)block * NTHREADS - t0 * per_tok), place = skipped + threadIdx.x, tl = place / (unsigned)per_tok;
  const long t = t0 + tl;
  const int k = (int)(place - tl * (unsigned)per_tok) * KV;
  const int wg_tokens = (int)min((long)((skipped + NTHREADS - 1) / (unsigned)per_tok) + 1, p.tokens - t0);   // >= 1
  float d[KV][PG_M], wk[KV];
  auto request = [&](long tt) {
#pragma unroll
    for (int j = 0; j < KV; ++j) load_row16<BF>(p.dist, (tt * p.K + k + j) * PG_M, d[j]);
#pragma unroll
    for (int j = 0; j < KV; ++j) wk[j] = p.weights ? p.weights[tt * p.K + k + j] : 1.0f;
  };
  if constexpr (CONV) request(min(t, p.tokens - 1));   // (under way while the first wave convolves)
  if constexpr (TOK) {
    const int n = wg_tokens * R;
    for (int e = threadIdx.x; e < n; e += NTHREADS) {
      const int tl = e / R, r = e - tl * R, i = r - p.H, set = i >= 2 * p.G ? 1 : 0;
      if (r < p.H) {
        tok_bias[e] = ld1<BF>(p.tok, (t0 + tl) * p.tok_stride + r) + p.tok_add[r];
      } else if constexpr (CONV) {
        if (set == 0) {   // (its lane has the second set's value too)
          const int at = (int)(t0 + tl);
          dw_chain_at<BF>(conv, at / conv.L, at % conv.L, conv.split + i, tok_bias[e], tok_bias[e + 2 * p.G]);
        }
      } else {
        tok_bias[e] = ld1<BF>(p.tail, (set * p.tokens + t0 + tl) * (2 * p.G) + i - set * 2 * p.G);
      }
    }
    __syncthreads();
  }
  if (t >= p.tokens) return;
  if constexpr (!CONV) request(t);
  // Outputs from the workgroup's first token on: a row is one scalar offset away from the row before, a thread's place one 32-bit offset.  (With a 64-bit
  // product a store, 109 v_mul_lo and 102 v_mad_u64, a quarter of the rate each, stood beside 360 multiply-adds: 8192 tokens x 256, fp32, 8 heads
  // 46 -> 38 us.)  Behind buffers; bf16 with gathered biases behind a scalar address, which suits its calls of few heads better, buffers and that, with
  // weights: 8192 x 256, 8 heads 32.8 and 31.8 us, 4096 x 1000, 2 heads 37.2 and 35.1, 4000 x 77, 3 heads 6.4 and 6.1 (the producers' biases in training, 8192 x 256
  // 33.4 and 34.4, fp32 62.5 and 64.0, 79.4 and 79.9, 7.8 and 7.9).
  constexpr int SZ = BF ? 2 : 4;
  const unsigned at_h = tl * (unsigned)(p.H * p.K) * SZ + (unsigned)k * SZ, at_g = tl * (unsigned)(p.G * p.K) * SZ + (unsigned)k * SZ;
  struct Rows {
    __amdgpu_buffer_rsrc_t buf;
    char* first;                  // row 0 of the workgroup's first token (FAR: the thread's place in row 0 of its token)
  };
  auto rows = [&](void* q, int per) __attribute__((always_inline)) {
    char* base = (char*)q + t0 * per * p.K * SZ;
    return Rows{__builtin_amdgcn_make_buffer_rsrc(base, 0, FAR ? 0u : (unsigned)(wg_tokens * per * p.K) * SZ, 0x00027000),
                FAR ? base + ((long)tl * per * p.K + k) * SZ : base};
  };
  auto put = [&](const Rows& to, unsigned at, int row, const float (&v)[KV]) __attribute__((always_inline)) {
    if constexpr (FAR) {
      st1<BF>(to.first, (long)row * p.K, v[0]);
    } else if constexpr (BF) {
      const unsigned two = KV == 2 ? (unsigned)f_to_bf16(v[0]) | ((unsigned)f_to_bf16(v[KV - 1]) << 16) : f_to_bf16(v[0]);
      char* q = to.first + (long)row * p.K * SZ + at;   // uniform, and the thread's
      if constexpr (TOK && KV == 2) __builtin_amdgcn_raw_buffer_store_b32(two, to.buf, at, row * p.K * SZ, 0);
      else if constexpr (TOK) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)two, to.buf, at, row * p.K * SZ, 0);
      else if constexpr (KV == 2) *(unsigned*)q = two;
      else *(uint16_t*)q = (uint16_t)two;
    } else if constexpr (KV == 2) {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64((u2){__float_as_uint(v[0]), __float_as_uint(v[1])}, to.buf, at, row * p.K * SZ, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), to.buf, at, row * p.K * SZ, 0);
    }
  };
  const Rows dt_rows = rows(p.dt, p.H), raw_rows = rows(RAW && p.dt_raw ? p.dt_raw : p.dt, p.H);
  const Rows bc_rows[4] = {rows(p.Bm, p.G), rows(p.Cm, p.G), rows(p.has_back ? p.Bb : p.Bm, p.G), rows(p.has_back ? p.Cb : p.Cm, p.G)};
  // the token's biases, all requested before the row loop (a load per row inside it would be waited for row by
  // row); bb: the reversed-order pair's bias of a B / C row
  float bv[PG_MAXR0], bb[PG_MAXR0];
  const float* bias = TOK ? tok_bias + (int)(t - t0) * R : p.bias + t * R;
#pragma unroll
  for (int r = 0; r < PG_MAXR0; ++r) {
    bv[r] = bias[min(r, R - 1)];
    bb[r] = bias[min(max(R0 + r - p.H, 0), R - 1)];
  }
#pragma unroll
  for (int r = 0; r < PG_MAXR0; ++r) {
    if (r < R0) {  // uniform
      // uniform: scalar loads, which the stores above do not stand in the way of (nothing here writes W)
      const __attribute__((address_space(4))) float* w = (const __attribute__((address_space(4))) float*)(uintptr_t)(p.W + r * PG_M);
      float s[KV], v[KV];
#pragma unroll
      for (int j = 0; j < KV; ++j) {
        s[j] = 0.0f;
#pragma unroll
        for (int m = 0; m < PG_M; ++m) s[j] = fmaf(w[m], d[j][m], s[j]);
        v[j] = s[j] + bv[r];
      }
      if (r < p.H) {
        if (p.weights) {  // uniform: dt = softplus(raw) * weight, raw kept for the backward
          if (BF) {
#pragma unroll
            for (int j = 0; j < KV; ++j) v[j] = bf16_to_f(f_to_bf16(v[j]));  // the saved value is what the backward differentiates
          }
          if (RAW) put(raw_rows, at_h, r, v);
#pragma unroll
          for (int j = 0; j < KV; ++j) v[j] = softplus_(v[j]) * wk[j];
        }
        put(dt_rows, at_h, r, v);
      } else {
        const bool isB = r < p.H + p.G;
        const int g = isB ? r - p.H : r - p.H - p.G;
        put(isB ? bc_rows[0] : bc_rows[1], at_g, g, v);
        if (p.has_back) {
#pragma unroll
          for (int j = 0; j < KV; ++j) v[j] = s[j] + bb[r];
          put(isB ? bc_rows[2] : bc_rows[3], at_g, g, v);
        }
      }
    }
  }
}

template <bool BF, int KV, bool TOK, bool RAW>
__global__ __launch_bounds__(NTHREADS) void k_pgen_fwd(PGenP p) {
  pgen_fwd<BF, KV, TOK, RAW, false, false>(p, DwConvP{}, blockIdx.x);
}
template <bool BF, bool TOK>
__global__ __launch_bounds__(NTHREADS) void k_pgen_fwd_far(PGenP p) {
  if (!p.weights || p.dt_raw) pgen_fwd<BF, 1, TOK, true, false, true>(p, DwConvP{}, blockIdx.x);
  else pgen_fwd<BF, 1, TOK, false, false, true>(p, DwConvP{}, blockIdx.x);
}

// What lies between a layer's first projections and its scan where no gradient is asked for, one launch: the generation above and,
// in the workgroups behind it, the convolutions of x.  The two took 9.5 and 5.6 us one after the other at a scene of 1024 tokens,
// 256 queries, 288 channels, each bound by its launch and a trip or two to memory; each token's 2G channels that the generation
// needs of the convolutions are computed by its own workgroup (13 inputs and 56 multiply-adds a channel).
template <int KV, int TL>
__global__ __launch_bounds__(NTHREADS) void k_conv_pgen(PGenP p, DwConvP c, int pgen_blocks) {
  warm_first<sizeof(PGenP) + sizeof(DwConvP)>();
  if ((int)blockIdx.x >= pgen_blocks) dw_chain_fwd<true, TL, false>(c, (long)((int)blockIdx.x - pgen_blocks) * NTHREADS + threadIdx.x);
  else pgen_fwd<true, KV, true, false, true, false>(p, c, blockIdx.x);
}
__global__ __launch_bounds__(NTHREADS) void k_conv_pgen_far(PGenP p, DwConvP c, int pgen_blocks) {
  if ((int)blockIdx.x >= pgen_blocks) dw_chain_fwd<true, 4, false>(c, (long)((int)blockIdx.x - pgen_blocks) * NTHREADS + threadIdx.x);
  else pgen_fwd<true, 1, true, false, true, true>(p, c, blockIdx.x);
}

// Gradient row r of token t: dt heads, then B groups, then C groups (`back`: the reversed-order pair, which
// exists for the B / C rows only).  Returns the element offset of (t, row, k = 0), or -1 when there is none.
struct GradRows {
  const void *ddt, *dB, *dC, *dBb, *dCb;
  int H, G, K;
  __device__ __forceinline__ const void* base(int r, bool back) const {
    if (r < H) return back ? nullptr : ddt;
    if (r < H + G) return back ? dBb : dB;
    if (r < H + 2 * G) return back ? dCb : dC;
    return nullptr;
  }
  __device__ __forceinline__ long offset(long t, int r) const {
    if (r < H) return (t * H + r) * K;
    if (r < H + G) return (t * G + (r - H)) * K;
    return (t * G + (r - H - G)) * K;
  }
};

// Loads without branches: a lane with nothing to read (no such row, k past the end) reads element 0 of `safe`
// -- any readable buffer of at least 16 bytes -- and the value is replaced by zero afterwards.  Branch-free
// loads can all be in flight together; a branch per load would serialise them.
template <bool BF>
__device__ __forceinline__ float ld1_or0(const void* p, long off, bool ok, const void* safe) {
  const float v = ld1<BF>(ok ? p : safe, ok ? off : 0);
  return ok ? v : 0.0f;
}
// Four consecutive elements p[off .. off + 3] for k .. k + 3 (k >= kend reads as zero).  `vec`: the address is
// aligned for one wide load and kend is a multiple of 4.
template <bool BF>
__device__ __forceinline__ f4 load4(const void* p, long off, int k, int kend, bool vec, const void* safe) {
  f4 r;
  if (vec) {  // uniform
    const bool ok = p != nullptr && k < kend;
    const void* q = ok ? p : safe;
    const long o = ok ? off : 0;
    if (BF) {
      const uint2 w = *(const uint2*)((const uint16_t*)q + o);
      r.x = __uint_as_float(w.x << 16); r.y = __uint_as_float(w.x & 0xffff0000u);
      r.z = __uint_as_float(w.y << 16); r.w = __uint_as_float(w.y & 0xffff0000u);
    } else {
      r = *(const f4*)((const float*)q + o);
    }
    if (!ok) r = (f4){0.0f, 0.0f, 0.0f, 0.0f};
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = ld1_or0<BF>(p, off + v, p != nullptr && k + v < kend, safe);
  }
  return r;
}

// d softplus(x) / dx with torch's threshold: 1 above 20
__device__ __forceinline__ float dsoftplus_(float x) { return x <= 20.0f ? sigmoidf_(x) : 1.0f; }

// Backward on the matrix cores (v_mfma_f32_16x16x4_f32; lane = (i = lane & 15, q = lane >> 4)).
// Workgroup = PG_TOK consecutive tokens, a wave owns PG_TOK / 4 of them and walks k in blocks of 16:
//   ddist^T (m x k) = W^T (m x r) g (r x k)   -- A: lane (m, q) = W[4s + q][m], B: lane (k, q) = g[4s + q][k0 + k];
//                                                the result lane (k, q) holds ddist[k0 + k][4q .. 4q + 3]: one wide store
//   dW (r x m)     += g (r x k) dist (k x m)  -- A: lane (r, q) = g[r][k0 + 4q + v], B: lane (m, q) = dist[k0 + 4q + v][m],
//                                                v = 0..3 (the order of k inside the sum is free)
//   dbias[r]        = sum_k g[r][k]           -- from the second layout, reduced over q at the end of the token.
// g of a B / C row is the sum of its forward-order and reversed-order gradients wherever the shared base row is
// differentiated; the two bias gradients stay apart.  HASW (dt = softplus(raw) * weight): g of a dt row is
// ddt * weight * softplus'(raw), and dweight[k] = sum_h ddt[h][k] softplus(raw[h][k]).
// FULLK: K is a multiple of 64, so no load or store needs a bound on k (pgen_pieces).
// PARTS: the bias gradients go to their producers and, summed, to bias_partial (issm_param_gen_bwd_part).  Known when compiled: asked at run time it
// cost every other call registers and its tail, 16384 tokens x 16 queries, bf16 27.7 -> 29.9 us, 4000 x 77, fp32 with weights 34.4 -> 37.7.
template <bool BF, bool FULLK, bool HASW, bool PARTS>
__global__ __launch_bounds__(NTHREADS, (BF || !HASW || !FULLK) ? 4 : 3) void k_pgen_bwd(PGenP p) {
  constexpr int KS = 128 / (BF ? 2 : 4);   // columns of a step: 128 bytes of a gradient row
  typedef typename std::conditional<BF, uint16_t, float>::type T;
  typedef typename std::conditional<BF, uint2, f4>::type T4;
  __shared__ float wred[4][16 * PG_M], bred[PARTS ? 4 : 1][16];
  // FULLK, each wave's own: a step's gradient rows and what goes with them (raw dt, reversed-order gradients; a row more for the lanes that have
  // none), its block of dist, the weights, and two tiles of effective gradients [row][k] in turn.
  __shared__ __align__(16) unsigned char srow[FULLK ? 4 : 1][2][FULLK ? (PG_MAXR0 + 1) * PG_LDR : 16];
  __shared__ __align__(16) unsigned char sd[FULLK ? 4 : 1][FULLK ? KS * PG_LDT * sizeof(T) : 16];
  __shared__ __align__(16) float sw[FULLK && HASW ? 4 : 1][FULLK && HASW ? KS : 4];
  __shared__ __align__(16) float sg[FULLK ? 4 : 1][FULLK ? 2 : 1][FULLK ? 16 * PG_LDT : 4];
  const int R0 = p.H + 2 * p.G, R = R0 + (p.has_back ? 2 * p.G : 0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, q = lane >> 4;
  const int K = p.K;
  const bool vec = (K & 3) == 0;
  const GradRows gr{p.ddt, p.dB, p.dC, p.has_back ? p.dBb : nullptr, p.has_back ? p.dCb : nullptr, p.H, p.G, K};
  float wA[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) wA[s] = (4 * s + q < R0) ? p.W[(4 * s + q) * PG_M + i] : 0.0f;
  // row-of-the-lane pointers: layout 2 (row i), layout 1 (rows 4s + q)
  const void* g2 = gr.base(i, false);
  const void* g2b = gr.base(i, true);
  const bool isdt2 = HASW && i < p.H && g2 != nullptr;
  const void *g1[3], *g1b[3];
  bool okg[3], okgb[3], isdt1[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    g1[s] = gr.base(4 * s + q, false);
    g1b[s] = gr.base(4 * s + q, true);
    okg[s] = g1[s] != nullptr;
    okgb[s] = g1b[s] != nullptr;
    isdt1[s] = HASW && 4 * s + q < p.H && okg[s];
  }
  const bool ok2 = g2 != nullptr, ok2b = g2b != nullptr;
  const bool any_back = gr.dBb != nullptr || gr.dCb != nullptr;  // uniform
  const f4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  auto widen = [](T4 w) -> f4 {
    if constexpr (BF) {
      return (f4){__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
                  __uint_as_float(w.y & 0xffff0000u)};
    } else {
      return w;
    }
  };
  auto widen1 = [](T w) -> float {
    if constexpr (BF) return __uint_as_float((unsigned)w << 16);
    else return w;
  };
  // one block of 16 k, operands already in registers (a / ab / rw2 / ww2: layout 2; x*, raw1, w1: layout 1)
  f4 accW = zero4;
  float bs = 0.0f, bsb = 0.0f, bsum = 0.0f;
  auto block = [&](f4 a, f4 ab, f4 rw2, f4 ww2, const float (&dv)[4], const float (&x)[3], const float (&xb)[3],
                   const float (&raw1)[3], float w1, T* ddst, float* dwdst, bool in_k) {
    if constexpr (HASW) {
      if (isdt2) {
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] *= ww2[v] * dsoftplus_(rw2[v]);
      }
    }
    bs += (a.x + a.y) + (a.z + a.w);
    bsb += (ab.x + ab.y) + (ab.z + ab.w);
#pragma unroll
    for (int v = 0; v < 4; ++v) accW = mfma4(a[v] + ab[v], dv[v], accW);
    float gx[3], dws = 0.0f;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      gx[s] = x[s];
      if constexpr (HASW) {
        if (isdt1[s]) {
          dws += x[s] * softplus_(raw1[s]);
          gx[s] = x[s] * w1 * dsoftplus_(raw1[s]);
        }
      }
      gx[s] += xb[s];
    }
    if constexpr (HASW) {
      if (dwdst != nullptr) {  // uniform
        dws += __shfl_xor(dws, 16, 64);
        dws += __shfl_xor(dws, 32, 64);
        if (q == 0 && in_k) *dwdst = dws;
      }
    }
    if (ddst != nullptr) {  // uniform
      f4 dd = zero4;
#pragma unroll
      for (int s = 0; s < 3; ++s) dd = mfma4(wA[s], gx[s], dd);
      if (in_k) {
        if constexpr (BF) {
          uint2 w;
          w.x = pack_bf16(dd.x, dd.y);
          w.y = pack_bf16(dd.z, dd.w);
          *(uint2*)ddst = w;
        } else {
          *(f4*)ddst = dd;
        }
      }
    }
  };

  constexpr int TPW = PG_TOK / 4;
  for (int ti = 0; ti < TPW; ++ti) {
    const long t = (long)blockIdx.x * PG_TOK + wave * TPW + ti;
    if (t >= p.tokens) break;  // wave-uniform
    const long o2 = i < R0 ? gr.offset(t, i) : 0;
    long o1[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) o1[s] = (4 * s + q < R0) ? gr.offset(t, 4 * s + q) : 0;
    bs = 0.0f;
    bsb = 0.0f;
    if constexpr (FULLK) {
      // Every operand is read once, in pieces of 16 bytes whose neighbours in memory are the neighbouring lanes' (eight lanes a gradient row,
      // the whole wave for dist), and goes through LDS that no other wave uses: the products need the rows with lane index =
      // gradient row (lane (i, q): row i, columns 16 u + 4 q .. + 3) and, from there, with lane index = column, and dist as operand columns.
      // (LDS instructions of one wave are carried out in order: a read sees the writes before it.)  A step's pieces are requested when the
      // step before has put its own into LDS; ddist takes dist's place there and leaves in the same pieces.  The rows read in the layout of
      // the products, 8 bytes a lane and 64 look-ups in the L1 an instruction, kept the look-ups busy 82 % of the time:
      // 8192 tokens x 256 queries, bf16, with weights, 53.4 -> 50.1 us, 234 MB at the rate of a copy (51.8 since it also leaves the producers their bias
      // gradients, for which an address goes to scratch before the loops and comes back behind them: 12 bytes a lane).
      // (The pieces' type promises the elements' alignment and no more: one wide access all the same.)
      typedef unsigned Piece __attribute__((ext_vector_type(4), aligned(2)));
      const T* nil = (const T*)p.dist;  // what a lane with no row reads (at least 64 * 16 elements long)
      const int piece = (lane & 7) * (16 / (int)sizeof(T));
      const T *pa[2], *px[2];
      bool oka[2], okx[2];
      int put[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = 8 * j + (lane >> 3);
        const bool isdt = HASW && row < p.H;
        const void *ga = gr.base(row, false), *gx = isdt ? p.dt_raw : gr.base(row, true);
        oka[j] = ga != nullptr;
        okx[j] = gx != nullptr && (!isdt || ga != nullptr);
        const long o = row < R0 ? gr.offset(t, row) + piece : 0;
        pa[j] = oka[j] ? (const T*)ga + o : nil;
        px[j] = okx[j] ? (const T*)gx + o : nil;
        put[j] = min(row, PG_MAXR0) * PG_LDR + (lane & 7) * 16;
      }
      const char* pd = (const char*)((const T*)p.dist + t * K * PG_M) + lane * 16;
      const float* pw = HASW ? p.weights + t * K + (lane & (KS - 1)) : nullptr;
      float* pdw = (HASW && p.dweights) ? p.dweights + t * K + 4 * q : nullptr;
      // (ddist: no buffer, no store, and no branch that would have the waits for the requests wait for the stores)
      const __amdgpu_buffer_rsrc_t dd_rows = __builtin_amdgcn_make_buffer_rsrc(
          p.ddist ? (T*)p.ddist + t * K * PG_M : nullptr, 0, p.ddist ? (unsigned)(K * PG_M * sizeof(T)) : 0u, 0x00027000);
      unsigned char *A = srow[wave][0], *X = srow[wave][1], *D = sd[wave];
      float* W = sw[wave];
      constexpr int LDD = PG_LDT * (int)sizeof(T);                 // row of dist, bytes
      constexpr int PR = PG_M * (int)sizeof(T) / 16;               // its pieces of 16
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      u4 ra[2], rx[2], rd[2];
      float rw = 0.0f;
      auto request = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          ra[j] = *(const Piece*)(pa[j] + (oka[j] ? k0 : 0));
          rx[j] = *(const Piece*)(px[j] + (okx[j] ? k0 : 0));
          rd[j] = *(const Piece*)(pd + (long)k0 * (PG_M * sizeof(T)) + 1024 * j);
        }
        if constexpr (HASW) rw = pw[k0];
      };
      request(0);
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): only requests of the loop's own steps count in it
      for (int k0 = 0; k0 < K; k0 += KS) {
        auto dist_piece = [&](int j) __attribute__((always_inline)) { return D + ((64 * j + lane) / PR) * LDD + (lane % PR) * 16; };
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          *(u4*)(A + put[j]) = ra[j];
          *(u4*)(X + put[j]) = rx[j];
          u2* d = (u2*)dist_piece(j);
          d[0] = rd[j].xy;
          d[1] = rd[j].zw;
        }
        if constexpr (HASW) W[lane & (KS - 1)] = rw;
        request(min(k0 + KS, K - KS));
#pragma unroll
        for (int u = 0; u < KS / 16; ++u) {
          float* S = sg[wave][u & 1];
          const int at = min(i, PG_MAXR0) * PG_LDR + (16 * u + 4 * q) * (int)sizeof(T);
          f4 a = ok2 ? widen(*(const T4*)(A + at)) : zero4;
          const f4 other = widen(*(const T4*)(X + at));
          const f4 ab = ok2b ? other : zero4;
          f4 pw4 = zero4;  // ddt * softplus(raw): the weight's gradient once summed over the heads
          if constexpr (HASW) {
            const f4 rw2 = *(const f4*)(W + 16 * u + 4 * q);
            if (isdt2) {
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                const float raw = other[v];
                const float tt = ex2(raw * LOG2E), uu = 1.0f + tt;
                const bool big = raw > 20.0f;  // torch's softplus threshold
                pw4[v] = a[v] * (big ? raw : LN2 * __builtin_amdgcn_logf(uu));
                a[v] *= rw2[v] * (big ? 1.0f : tt * __builtin_amdgcn_rcpf(uu));
              }
            }
          }
          bs += (a.x + a.y) + (a.z + a.w);
          bsb += (ab.x + ab.y) + (ab.z + ab.w);
          const f4 g = a + ab;
          *(f4*)(S + i * PG_LDT + 4 * q) = g;
          float dv[4], x[3];
          const T* dist = (const T*)(D + 16 * u * LDD);
#pragma unroll
          for (int v = 0; v < 4; ++v) dv[v] = widen1(dist[(4 * q + v) * PG_LDT + i]);
#pragma unroll
          for (int s = 0; s < 3; ++s) x[s] = S[(4 * s + q) * PG_LDT + i];
#pragma unroll
          for (int v = 0; v < 4; ++v) accW = mfma4(g[v], dv[v], accW);
          f4 dd = zero4;
#pragma unroll
          for (int s = 0; s < 3; ++s) dd = mfma4(wA[s], x[s], dd);
          T4* dst = (T4*)(D + (16 * u + i) * LDD + 4 * q * (int)sizeof(T));
          if constexpr (BF) *dst = make_uint2(pack_bf16(dd.x, dd.y), pack_bf16(dd.z, dd.w));
          else *dst = dd;
          if constexpr (HASW) {
            if (pdw != nullptr) {  // uniform: sum over the rows = over the 16 lanes that share q
#pragma unroll
              for (int v = 0; v < 4; ++v) pw4[v] = row_sum16_(pw4[v]);
              if (i == 15) *(f4*)(pdw + k0 + 16 * u) = pw4;
            }
          }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u2* d = (const u2*)dist_piece(j);
          const u2 lo = d[0], hi = d[1];
          __builtin_amdgcn_raw_buffer_store_b128((u4){lo.x, lo.y, hi.x, hi.y}, dd_rows,
                                                 (unsigned)(k0 * PG_M * (int)sizeof(T) + 1024 * j + lane * 16), 0, 0);
        }
      }
    } else {
      const void* safe = p.W;
      for (int k0 = 0; k0 < K; k0 += 16) {
        const int kq = k0 + 4 * q;
        const bool in = k0 + i < K;
        const f4 a = load4<BF>(g2, o2 + kq, kq, K, vec, safe);
        const f4 ab = any_back ? load4<BF>(g2b, o2 + kq, kq, K, vec, safe) : zero4;
        f4 rw2 = zero4, ww2 = zero4;
        float dv[4], x[3], xb[3], raw1[3], w1 = 0.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) dv[v] = ld1_or0<BF>(p.dist, (t * K + kq + v) * PG_M + i, kq + v < K, safe);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          x[s] = ld1_or0<BF>(g1[s], o1[s] + k0 + i, in && okg[s], safe);
          xb[s] = any_back ? ld1_or0<BF>(g1b[s], o1[s] + k0 + i, in && okgb[s], safe) : 0.0f;
          raw1[s] = HASW ? ld1_or0<BF>(p.dt_raw, o1[s] + k0 + i, in && isdt1[s], safe) : 0.0f;
        }
        if constexpr (HASW) {
          rw2 = load4<BF>(isdt2 ? p.dt_raw : nullptr, o2 + kq, kq, K, vec, safe);
          ww2 = load4<false>(p.weights, t * K + kq, kq, K, vec, safe);
          w1 = ld1_or0<false>(p.weights, t * K + k0 + i, in, safe);
        }
        block(a, ab, rw2, ww2, dv, x, xb, raw1, w1,
              p.ddist ? (T*)p.ddist + (t * K + k0 + i) * PG_M + 4 * q : nullptr,
              (HASW && p.dweights) ? p.dweights + t * K + k0 + i : nullptr, in);
      }
    }
    bs += __shfl_xor(bs, 16, 64);
    bs += __shfl_xor(bs, 32, 64);
    bsb += __shfl_xor(bsb, 16, 64);
    bsb += __shfl_xor(bsb, 32, 64);
    if (p.dbias && q == 0 && i < R0) {
      p.dbias[t * R + i] = bs;
      if (p.has_back && i >= p.H) p.dbias[t * R + R0 + (i - p.H)] = bsb;
    }
    if constexpr (PARTS) {
      bsum += bs;
      auto io = [](float v) -> T {
        if constexpr (BF) return f_to_bf16(v);
        else return v;
      };
      if (q == 0 && i < p.H) ((T*)p.dtok)[t * p.dtok_stride + i] = io(bs);
      if (q == 0 && i >= p.H && i < R0) {
        T* to = (T*)p.dtail + t * (2 * p.G) + (i - p.H);
        to[0] = io(bs);
        to[p.tokens * (2 * p.G)] = io(bsb);
      }
    }
  }
  // dW partial of the workgroup: the four waves in order.  Lane (m, q) holds rows 4q .. 4q + 3 of column m.
#pragma unroll
  for (int v = 0; v < 4; ++v) wred[wave][(4 * q + v) * PG_M + i] = accW[v];
  if constexpr (PARTS)
    if (q == 0) bred[wave][i] = bsum;
  __syncthreads();
  for (int e = threadIdx.x; e < R0 * PG_M; e += NTHREADS)
    p.dw_partial[(long)blockIdx.x * R0 * PG_M + e] = (wred[0][e] + wred[1][e]) + (wred[2][e] + wred[3][e]);
  if constexpr (PARTS) {
    const int r = threadIdx.x;
    if (r < R0) p.bias_partial[(long)blockIdx.x * R0 + r] = (bred[0][r] + bred[1][r]) + (bred[2][r] + bred[3][r]);
  }
}

// dW = fixed-order sum of the per-workgroup partials: one workgroup per entry of dW; the workgroups after those sum
// one column of dbias over the tokens each (same tree, so both are reproducible)
__global__ __launch_bounds__(NTHREADS) void k_pgen_dw(PGenP p) {
  __shared__ float red[NTHREADS];
  const int n = (p.H + 2 * p.G) * PG_M;
  const int c = blockIdx.x;
  float a0 = 0.0f, a1 = 0.0f;
  if (c < n) {
    int b = threadIdx.x;
    for (; b + NTHREADS < p.nblocks; b += 2 * NTHREADS) {
      a0 += p.dw_partial[(long)b * n + c];
      a1 += p.dw_partial[(long)(b + NTHREADS) * n + c];
    }
    if (b < p.nblocks) a0 += p.dw_partial[(long)b * n + c];
  } else {
    const int R = p.H + 2 * p.G + (p.has_back ? 2 * p.G : 0), r = c - n;
    long t = threadIdx.x;
    // latency: the adds are a chain in a fixed order, but the loads of eight rounds travel together (8.3 -> 6.9 us at 8192
    // tokens)
#pragma unroll 8
    for (; t + NTHREADS < p.tokens; t += 2 * NTHREADS) {
      a0 += p.dbias[t * R + r];
      a1 += p.dbias[(t + NTHREADS) * R + r];
    }
    if (t < p.tokens) a0 += p.dbias[t * R + r];
  }
  red[threadIdx.x] = a0 + a1;
  __syncthreads();
#pragma unroll
  for (int w = NTHREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (c < n) p.dW[c] = red[0];
    else p.dbias_sum[c - n] = red[0];
  }
}

int pgen_bwd_blocks(long tokens) { return (int)((tokens + PG_TOK - 1) / PG_TOK); }

// adjacent outputs go out as one store: K a multiple of the group and every output 16-byte aligned
static int pgen_group(const PGenP& p) {
  uintptr_t bits = 0;
  for (const void* q : {(const void*)p.dt, (const void*)p.dt_raw, (const void*)p.Bm, (const void*)p.Cm, (const void*)p.Bb,
                        (const void*)p.Cb})
    bits |= (uintptr_t)q;
  const bool al = (bits & 15) == 0;
  // (four adjacent k per thread, 8-byte bf16 stores, measured slower: 42 us against 39 at 8192 tokens x 256)
  return (p.K % 2 == 0 && al) ? 2 : 1;
}
// Whether the rows of the two tokens that a workgroup of so many queries may have reach beyond 31-bit byte offsets
static bool pgen_far(const PGenP& p) { return 2L * std::max(p.H, p.G) * p.K * (p.dtype ? 2 : 4) >= 1L << 31; }
static size_t pgen_lds(const PGenP& p, int per_tok) {
  const int R = p.H + (p.has_back ? 4 : 2) * p.G;
  return p.bias ? 0 : ((NTHREADS - 1) / per_tok + 2) * (size_t)R * sizeof(float);   // at most 23 KB
}

int launch_pgen_fwd(const PGenP& p, hipStream_t st) {
  const bool far = pgen_far(p);
  const int kv = far ? 1 : pgen_group(p), per_tok = (p.K + kv - 1) / kv;
  const unsigned blocks = (unsigned)((p.tokens * per_tok + NTHREADS - 1) / NTHREADS);
  const size_t lds = pgen_lds(p, per_tok);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(blocks), dim3(NTHREADS), lds, st, p); };
  if (far) {
    if (p.dtype) p.bias ? go(&k_pgen_fwd_far<true, false>) : go(&k_pgen_fwd_far<true, true>);
    else p.bias ? go(&k_pgen_fwd_far<false, false>) : go(&k_pgen_fwd_far<false, true>);
    return (int)hipGetLastError();
  }
  const bool raw = !p.weights || p.dt_raw;
  auto forms = [&](auto two, auto one, auto two_only, auto one_only) { raw ? go(kv == 2 ? two : one) : go(kv == 2 ? two_only : one_only); };
  if (p.bias) {
    if (p.dtype) forms(&k_pgen_fwd<true, 2, false, true>, &k_pgen_fwd<true, 1, false, true>, &k_pgen_fwd<true, 2, false, false>, &k_pgen_fwd<true, 1, false, false>);
    else forms(&k_pgen_fwd<false, 2, false, true>, &k_pgen_fwd<false, 1, false, true>, &k_pgen_fwd<false, 2, false, false>, &k_pgen_fwd<false, 1, false, false>);
  } else {
    if (p.dtype) forms(&k_pgen_fwd<true, 2, true, true>, &k_pgen_fwd<true, 1, true, true>, &k_pgen_fwd<true, 2, true, false>, &k_pgen_fwd<true, 1, true, false>);
    else forms(&k_pgen_fwd<false, 2, true, true>, &k_pgen_fwd<false, 1, true, true>, &k_pgen_fwd<false, 2, true, false>, &k_pgen_fwd<false, 1, true, false>);
  }
  return (int)hipGetLastError();
}

int launch_conv_pgen(const DwConvP& c, const PGenP& p, hipStream_t st) {
  const bool far = pgen_far(p);
  const int kv = far ? 1 : pgen_group(p), per_tok = (p.K + kv - 1) / kv;
  const long gen = (p.tokens * per_tok + NTHREADS - 1) / NTHREADS;
  // tokens a thread of the convolutions: as few as leave two waves a SIMD (see there)
  auto items = [&](int tokens) { return (long)c.B * ((c.L + tokens - 1) / tokens) * c.split; };
  const int tl = far ? 4 : items(16) >= 2048 * 64 ? 16 : items(8) >= 2048 * 64 ? 8 : 4;
  const long conv = (items(tl) + NTHREADS - 1) / NTHREADS;
  if (gen + conv > 0x7fffffff) return (int)hipErrorInvalidValue;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)(gen + conv)), dim3(NTHREADS), pgen_lds(p, per_tok), st, p, c, (int)gen); };
  auto form = [&](auto two, auto one) { kv == 2 ? go(two) : go(one); };
  if (far) go(&k_conv_pgen_far);
  else if (tl == 16) form(&k_conv_pgen<2, 16>, &k_conv_pgen<1, 16>);
  else if (tl == 8) form(&k_conv_pgen<2, 8>, &k_conv_pgen<1, 8>);
  else form(&k_conv_pgen<2, 4>, &k_conv_pgen<1, 4>);
  return (int)hipGetLastError();
}

// Whether the backward goes by whole steps of 64 queries, of which it requests the first unasked, a token's ddist behind a buffer: 32-bit offsets, and
// whole dwords to store
static bool pgen_pieces(const PGenP& p) { return p.K > 0 && p.K % 64 == 0 && p.K < 1 << 24 && ((uintptr_t)p.ddist & 3) == 0; }
template <bool BF, bool HASW>
static void pgen_bwd_launch(const PGenP& p, hipStream_t st) {
  const dim3 g((unsigned)p.nblocks), b(NTHREADS);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, b, 0, st, p); };
  if (pgen_pieces(p)) p.dtail ? go(&k_pgen_bwd<BF, true, HASW, true>) : go(&k_pgen_bwd<BF, true, HASW, false>);
  else p.dtail ? go(&k_pgen_bwd<BF, false, HASW, true>) : go(&k_pgen_bwd<BF, false, HASW, false>);
}

int launch_pgen_bwd(const PGenP& p, hipStream_t st) {
  const int R0 = p.H + 2 * p.G;
  if (p.dtype) {
    if (p.weights) pgen_bwd_launch<true, true>(p, st);
    else pgen_bwd_launch<true, false>(p, st);
  } else {
    if (p.weights) pgen_bwd_launch<false, true>(p, st);
    else pgen_bwd_launch<false, false>(p, st);
  }
  int e = (int)hipGetLastError();
  if (e || !p.dW) return e;
  const int R = R0 + (p.has_back ? 2 * p.G : 0);
  hipLaunchKernelGGL(k_pgen_dw, dim3(R0 * PG_M + (p.dbias_sum ? R : 0)), dim3(NTHREADS), 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
