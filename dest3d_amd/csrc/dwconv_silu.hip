// Depthwise 7-tap convolution along the token order + SiLU, on (B, L, C) tensors as they are (gfx950).
//
// DEST's PointLiteConv (models/dest_module.py:400-423) is nn.Conv1d(C, C, 7, padding=3, groups=C) + SiLU applied
// to feature.transpose(1, 2).  A library convolution sees (B, C, L) and pays for two transposes and an
// im2col-style lowering; here channels stay innermost (lanes run over c: every access is coalesced) and a thread
// owns DW_TL consecutive tokens of one channel, with the 3 + 3 halo rows in registers.  `nsets` weight sets are applied in one pass:
//   pre[s][b][l][c] = bias[s][c] + sum_j w[s][c][j] in_s[b][l + j - 3][c]      (zero outside [0, L))
//   y[s] = pre[s] * sigmoid(pre[s])
// with in_s = u for every set, or -- `chain` -- in_0 = u and in_1 = y[0]: the module's reversed-order branch convolves the
// forward-order branch's OUTPUT (dest_module.py:530 reassigns xbc = key_conv(xbc) before :534 calls key_conv_back on it).
// The chained kernels take a 6 + 6 halo of u so that y[0] is at hand on the 3 + 3 halo the second convolution needs, in tiles through LDS
// (y[0] outside [0, L) is the second convolution's zero padding, not the first one applied to padding).
// The backward reads dy and the saved pre: dpre = dy * sigmoid(pre) * (1 + pre * (1 - sigmoid(pre))),
//   du[b][l][c] = sum_s sum_j w[s][c][j] dpre[s][b][l + 3 - j][c],
//   dw[s][c][j] = sum_{b,l} dpre[s][b][l][c] u[b][l + j - 3][c],   dbias[s][c] = sum_{b,l} dpre[s][b][l][c],
// the last two as partials (one per (b, token tile)) summed in fixed order by a second kernel.
// Memory moves 24 MB forward and 29 backward at 8 x 1024 tokens, 290 channels, bf16, 5 and 6 us; the exponentials and the two rows of seven
// products a value come to about as much, and a launch's waves are there at once, so that neither hides all of the other: 8.5 and 14.6 us
// chained.  Arithmetic is fp32.
#include <algorithm>

#include "dwconv_dev.h"

namespace issm {

// Tokens per thread of the kernels that are not chained, DW_TL.  Backward: 16.  Forward: the most of 16, 8 and 4 that makes two waves a SIMD: one
// scene of 1024 tokens makes 290 waves of 16 (9.4, 7.7 and 5.5 us with 16, 8 and 4).
// Tokens per tile of the chained ones.  Backward: 64 (32: 17.3 us with half more of the sums for the parts; 64: 17.2, of which 2 went with the
// sums' LDS that left a CU four workgroups of five).  Forward: 64, or 16 where that makes fewer than 1024 workgroups (and more: launch_dwconv_fwd).
constexpr int DW_BWD = 16, DW_CHAIN_BWD = 64;

template <bool BF, int S, int DW_TL>
__global__ __launch_bounds__(NTHREADS) void k_dwconv_fwd(DwConvP p) {
  int b, l0, c;
  if (!dw_item<DW_TL>(p, (long)blockIdx.x * NTHREADS + threadIdx.x, p.C, b, l0, c)) return;
  float w[S][DW_TAPS], bias[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + c) * DW_TAPS + j];
    bias[s] = p.bias[(long)s * p.C + c];
  }
  const long ub = (long)b * p.u_bs + c;
  // rows outside [0, L) read row 0 or L - 1 and are replaced by zero: loads without branches stay in flight together
  auto u_at = [&](int l) -> float {
    const float v = dw_ld<BF>(p.u, ub + (long)min(max(l, 0), p.L - 1) * p.u_ls);
    return (l >= 0 && l < p.L) ? v : 0.0f;
  };
  float ub_[DW_TL + DW_TAPS - 1];  // u[l0 - 3 .. l0 + DW_TL + 2]: every load is issued before the first use
#pragma unroll
  for (int j = 0; j < DW_TL + DW_TAPS - 1; ++j) ub_[j] = u_at(l0 + j - 3);
#pragma unroll
  for (int i = 0; i < DW_TL; ++i) {
    const int l = l0 + i;
    if (l < p.L) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        float a = bias[s];
#pragma unroll
        for (int j = 0; j < DW_TAPS; ++j) a = fmaf(w[s][j], ub_[i + j], a);
        const long o = (((long)s * p.B + b) * p.L + l) * p.C + c;
        if (BF) a = bf16_to_f(f_to_bf16(a));  // the saved pre-activation is what the backward differentiates
        dw_st<BF>(p.pre, o, a);
        const float yv = a * sigmoidf_(a);
        if (p.split > 0) {  // uniform: channels [0, split) and [split, C) go to two dense tensors
          const long row = ((long)s * p.B + b) * p.L + l;
          if (c < p.split) dw_st<BF>(p.y, row * p.split + c, yv);
          else dw_st<BF>(p.y_tail, row * (p.C - p.split) + (c - p.split), yv);
        } else {
          dw_st<BF>(p.y, o, yv);
        }
      }
    }
  }
}

// partial layout: [(b * ntile + tile)][s][j (0..6: taps, 7: bias)][c]
template <bool BF, int S>
__global__ __launch_bounds__(NTHREADS) void k_dwconv_bwd(DwConvP p) {
  constexpr int DW_TL = DW_BWD;
  int b, l0, c;
  if (!dw_item<DW_TL>(p, (long)blockIdx.x * NTHREADS + threadIdx.x, p.C, b, l0, c)) return;
  float w[S][DW_TAPS];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + c) * DW_TAPS + j];
  const long ub = (long)b * p.u_bs + c;
  constexpr int W = DW_TL + DW_TAPS - 1;
  float ub_[W], dyb[S][W], prb[S][W];  // rows l0 - 3 .. l0 + DW_TL + 2, loaded before the first use
#pragma unroll
  for (int j = 0; j < W; ++j) {
    // rows outside [0, L) read row 0 or L - 1 and are replaced by zero: loads without branches stay in flight together
    const int l = l0 + j - 3, lc = min(max(l, 0), p.L - 1);
    const bool in = l >= 0 && l < p.L;
    const float uv = dw_ld<BF>(p.u, ub + (long)lc * p.u_ls);
    ub_[j] = in ? uv : 0.0f;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const long o = ((long)b * p.L + lc) * p.C + c;
      // with a split the gradient arrives as the two dense tensors of the forward: which one a lane reads is chosen
      // by selecting the address, not by a branch (an absent tensor reads `pre` and counts as zero), so that all
      // loads of the thread stay in flight together
      const bool head = p.split <= 0 || c < p.split;
      const void* src = head ? p.dy[s] : p.dy_tail[s];
      const long row = (long)b * p.L + lc;
      long off = o;
      if (p.split > 0) off = head ? row * p.split + c : row * (p.C - p.split) + (c - p.split);  // uniform condition
      const bool have = src != nullptr;
      const float dyv = dw_ld<BF>(have ? src : p.pre, have ? off : o);
      const float pv = dw_ld<BF>(p.pre, (long)s * p.B * p.L * p.C + o);
      dyb[s][j] = (in && have) ? dyv : 0.0f;
      prb[s][j] = in ? pv : 0.0f;
    }
  }
  // dpre in place of dy
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const float x = prb[s][j], sg = sigmoidf_(x);
      dyb[s][j] *= sg * (1.0f + x * (1.0f - sg));
    }
  float gw[S][DW_TAPS], gb[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    gb[s] = 0.0f;
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) gw[s][j] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < DW_TL; ++i) {
    const int l = l0 + i;
    if (l < p.L) {
      float du = 0.0f;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        // u[l] feeds pre[l + 3 - j] through tap j: buffer slot i + 6 - j
#pragma unroll
        for (int j = 0; j < DW_TAPS; ++j) du = fmaf(w[s][j], dyb[s][i + DW_TAPS - 1 - j], du);
        const float d0 = dyb[s][i + 3];  // dpre[s][l]
        gb[s] += d0;
#pragma unroll
        for (int j = 0; j < DW_TAPS; ++j) gw[s][j] = fmaf(d0, ub_[i + j], gw[s][j]);
      }
      if (p.du) dw_st<BF>(p.du, (long)b * p.du_bs + (long)l * p.du_ls + c, du);
    }
  }
  const int ntile = (p.L + DW_TL - 1) / DW_TL;
  const long row = (long)b * ntile + l0 / DW_TL;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    float* dst = p.partial + ((row * S + s) * 8) * p.C + c;
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) dst[(long)j * p.C] = gw[s][j];
    dst[(long)DW_TAPS * p.C] = gb[s];
  }
}

// ---- chained pair: set 1 convolves set 0's output (rounded to the I/O dtype, as it is stored)
// A thread to DW_TL tokens of a channel: rows far apart (the tiles below address theirs in 32 bits), and fp32 whose rows no cache holds (launch_dwconv_fwd)
template <bool BF, int DW_TL>
__global__ __launch_bounds__(NTHREADS) void k_dwconv_chain_fwd_threads(DwConvP p) {
  dw_chain_fwd<BF, DW_TL, true>(p, (long)blockIdx.x * NTHREADS + threadIdx.x);
}

constexpr int DW_CH = 32, DW_RUNS = NTHREADS / DW_CH, DW_HALO = DW_TAPS - 1;

// A workgroup's tile of T tokens x 32 channels and the thread's channel of it; the channels in front of the split and behind it have tiles of
// their own.
template <int T>
struct DwTile {
  int cl, run, row, b, l0, width, part, c;   // row: of the tiles along the tokens; width, part: channels of the split's side, the thread's among them
  bool head, have;
  __device__ __forceinline__ DwTile(const DwConvP& p) {
    cl = threadIdx.x & (DW_CH - 1);
    run = threadIdx.x / DW_CH;
    const int split = p.split > 0 ? p.split : p.C, htiles = (split + DW_CH - 1) / DW_CH, ctiles = htiles + (p.C - split + DW_CH - 1) / DW_CH;
    const int ntile = (p.L + T - 1) / T, wg = xcd_remap(blockIdx.x, gridDim.x);   // (an XCD's workgroups share rows' memory lines)
    const int ct = wg % ctiles;
    row = wg / ctiles;
    b = row / ntile;
    l0 = row % ntile * T;
    head = ct < htiles;   // uniform
    width = head ? split : p.C - split;
    part = (head ? ct : ct - htiles) * DW_CH + cl;
    c = head ? part : split + part;
    have = part < width;
  }
};
static unsigned dw_tiles(const DwConvP& p, int tokens) {
  const int split = p.split > 0 ? p.split : p.C;
  return (unsigned)p.B * ((p.L + tokens - 1) / tokens) * ((split + DW_CH - 1) / DW_CH + (p.C - split + DW_CH - 1) / DW_CH);
}
// Whether a tile's rows (76, or 140 of 2-byte values) are within 31-bit byte offsets
static bool dw_near(const DwConvP& p) { return std::max(std::max(p.u_ls, p.du ? p.du_ls : 0L), (long)p.C) < 1L << 22; }

// Rows from .. to - 1 behind a buffer: what lies outside them or the channels reads zero and is not stored, an addition an access where a pointer, a
// clamped row and the zero took ten.
template <bool BF>
struct DwRows {
  typedef typename std::conditional<BF, uint16_t, float>::type IO;
  __amdgpu_buffer_rsrc_t buf;
  unsigned first, ls;   // bytes: the lane's channel in row `from`, a row
  // q: row 0 of the sequence, `wide` channels of rows `ls` elements apart
  __device__ __forceinline__ DwRows(const void* q, long ls_, int wide, int from, int to, int channel, bool have) {
    ls = (unsigned)(ls_ * (long)sizeof(IO));
    buf = __builtin_amdgcn_make_buffer_rsrc((char*)const_cast<void*>(q) + (long)from * ls_ * (long)sizeof(IO), 0,
                                            q ? (unsigned)(((long)(to - from - 1) * ls_ + wide) * (long)sizeof(IO)) : 0u, 0x00027000);
    first = have ? (unsigned)channel * (unsigned)sizeof(IO) : 0x80000000u;
  }
  __device__ __forceinline__ float load(int row) const {   // row: relative to `from`
    const unsigned o = first + (unsigned)row * ls;
    if constexpr (BF) return bf16_to_f(__builtin_amdgcn_raw_buffer_load_b16(buf, o, 0, 0));
    else return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, o, 0, 0));
  }
  __device__ __forceinline__ void store(int row, float v) const {
    const unsigned o = first + (unsigned)row * ls;
    if constexpr (BF) __builtin_amdgcn_raw_buffer_store_b16(f_to_bf16(v), buf, o, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), buf, o, 0, 0);
  }
};
// a pointer `n` elements on, null if null
template <typename IO>
__device__ __forceinline__ const void* dw_at(const void* q, long n) {
  return q ? (const IO*)q + n : nullptr;
}

// Thread = channel and one of eight runs of rows; u and y[0] go through LDS, so that the halo of 6 + 6 rows is loaded and convolved once a
// workgroup, not once a thread.  290 channels, bf16, us, with a thread to 16, 8 or 4 tokens and now: 1 x 1024 tokens 4.8 and 3.7, 8 x 1024 14.8 and 8.5,
// 16 x 4096 67.8 and 41.2.
template <bool BF, int T>
__global__ __launch_bounds__(NTHREADS) void k_dwconv_chain_fwd(DwConvP p) {
  constexpr int CH = DW_CH, RUNS = DW_RUNS, HALO = DW_HALO, N0 = T + HALO, N1 = N0 + HALO;
  constexpr int K1 = (N1 + RUNS - 1) / RUNS, K0 = (N0 + RUNS - 1) / RUNS, K = T / RUNS;   // rows a thread
  typedef typename std::conditional<BF, uint16_t, float>::type IO;
  __shared__ float us[RUNS * (K1 > K0 ? K1 : K0) + HALO][CH], y0[RUNS * K0][CH];   // rows l0 - 6 .., l0 - 3 ..
  const DwTile<T> t(p);
  const int cl = t.cl, run = t.run, l0 = t.l0, cc = min(t.c, p.C - 1);
  float w[2][DW_TAPS], bias[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + cc) * DW_TAPS + j];
    bias[s] = p.bias[(long)s * p.C + cc];
  }
  const int from = max(l0 - HALO, 0), to = min(l0 + T + HALO, p.L), end = min(l0 + T, p.L);
  const DwRows<BF> u(dw_at<IO>(p.u, (long)t.b * p.u_bs), p.u_ls, p.C, from, to, t.c, t.have);
  float uv[K1];
#pragma unroll
  for (int k = 0; k < K1; ++k) uv[k] = u.load(l0 - HALO - from + run + RUNS * k);
#pragma unroll
  for (int k = 0; k < K1; ++k) us[run + RUNS * k][cl] = uv[k];
  __syncthreads();
  const long seq = (long)p.L * p.C, part_seq = (long)p.L * t.width;
  auto out = [&](int s, bool y) __attribute__((always_inline)) {
    return y ? DwRows<BF>(dw_at<IO>(t.head ? p.y : p.y_tail, ((long)s * p.B + t.b) * part_seq), t.width, t.width, l0, end, t.part, t.have)
             : DwRows<BF>(dw_at<IO>(p.pre, ((long)s * p.B + t.b) * seq), p.C, p.C, l0, end, t.c, t.have);
  };
  {
    const DwRows<BF> pre = out(0, false), y = out(0, true);
    float v[K0 + HALO];
#pragma unroll
    for (int k = 0; k < K0 + HALO; ++k) v[k] = us[run * K0 + k][cl];
#pragma unroll
    for (int k = 0; k < K0; ++k) {
      const int j = run * K0 + k, l = l0 - HALO / 2 + j;
      float a = bias[0];
#pragma unroll
      for (int i = 0; i < DW_TAPS; ++i) a = fmaf(w[0][i], v[k + i], a);
      a = dw_round<BF>(a);   // the saved pre-activation is what the backward differentiates
      const float yv = dw_round<BF>(a * sigmoidf_(a));
      pre.store(l - l0, a);   // (rows outside the tile are dropped)
      y.store(l - l0, yv);
      y0[j][cl] = l >= 0 && l < p.L ? yv : 0.0f;
    }
  }
  __syncthreads();
  const DwRows<BF> pre = out(1, false), y = out(1, true);
  float v[K + HALO];
#pragma unroll
  for (int k = 0; k < K + HALO; ++k) v[k] = y0[run * K + k][cl];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float a = bias[1];
#pragma unroll
    for (int i = 0; i < DW_TAPS; ++i) a = fmaf(w[1][i], v[k + i], a);
    a = dw_round<BF>(a);
    pre.store(run * K + k, a);
    y.store(run * K + k, a * sigmoidf_(a));
  }
}

// Workgroup = DW_CHAIN_BWD tokens x 32 channels; thread = channel and one of eight runs of rows.  What either convolution's gradient reads from
// rows around it -- dpre[1], then dpre[0], y[0], u -- goes through LDS, so that the halo of 6 + 6 rows is loaded and differentiated once a
// workgroup.  290 channels, bf16, us, with a thread to 8 tokens and now, the parts' sums included: 1 x 1024 tokens 9.7 and 8.1, 8 x 1024 28.4 and 14.7,
// 16 x 4096 190 and 70; the parts are an eighth as many.
template <bool BF, bool FAR>   // FAR: rows too far apart for buffers
__global__ __launch_bounds__(NTHREADS) void k_dwconv_chain_bwd(DwConvP p) {
  constexpr int T = DW_CHAIN_BWD, CH = DW_CH, RUNS = DW_RUNS, HALO = DW_HALO;
  constexpr int N0 = T + HALO, N1 = N0 + HALO;                                       // rows of set 0's arrays, of set 1's
  constexpr int K1 = (N1 + RUNS - 1) / RUNS, K0 = (N0 + RUNS - 1) / RUNS, K = T / RUNS;   // rows a thread
  typedef typename std::conditional<BF, uint16_t, float>::type IO;
  // dpre[1] on rows l0 - 6 .., dpre[0], y[0] and u on rows l0 - 3 ..; room for all rows of all threads, the last ones' are not read
  __shared__ float d1[RUNS * K1][CH], d0[RUNS * K0][CH];
  __shared__ IO y0[RUNS * K0][CH], us[RUNS * K0][CH];
  static_assert(RUNS * K1 >= RUNS * K0 + HALO && RUNS * K1 >= NTHREADS / 64 * 16, "rows that are read, the sums of the waves");
  float(&red)[RUNS * K1][CH] = d1;   // (the sums of the waves, when it has been read)
  const DwTile<T> t(p);
  const int cl = t.cl, run = t.run, l0 = t.l0, cc = min(t.c, p.C - 1);
  float w[2][DW_TAPS];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j < DW_TAPS; ++j) w[s][j] = p.w[((long)s * p.C + cc) * DW_TAPS + j];
  auto in = [&](int l) { return l >= 0 && l < p.L; };
  // every load is issued before the first use; an absent gradient counts as zero
  const int from = max(l0 - HALO, 0), to = min(l0 + T + HALO, p.L);
  struct Rows {
    DwRows<BF> near;
    const void* base;
    long ls;
    int channel;
  };
  auto rows = [&](const void* q, long ls, int wide, int channel) __attribute__((always_inline)) {
    return Rows{DwRows<BF>(FAR ? nullptr : q, ls, wide, from, to, channel, t.have), q, ls, channel};
  };
  auto load = [&](const Rows& r, int l) __attribute__((always_inline)) -> float {
    if constexpr (FAR) {
      const bool ok = in(l) && t.have && r.base;
      const float v = dw_ld<BF>(ok ? r.base : p.pre, ok ? l * r.ls + r.channel : 0);
      return ok ? v : 0.0f;
    } else {
      return r.near.load(l - from);
    }
  };
  const long seq = (long)p.L * p.C, part_seq = (long)p.L * t.width;
  const Rows dy1 = rows(dw_at<IO>(t.head ? p.dy[1] : p.dy_tail[1], t.b * part_seq), t.width, t.width, t.part),
             dy0 = rows(dw_at<IO>(t.head ? p.dy[0] : p.dy_tail[0], t.b * part_seq), t.width, t.width, t.part),
             pre1 = rows(dw_at<IO>(p.pre, (p.B + t.b) * seq), p.C, p.C, t.c), pre0 = rows(dw_at<IO>(p.pre, t.b * seq), p.C, p.C, t.c),
             u = rows(dw_at<IO>(p.u, (long)t.b * p.u_bs), p.u_ls, p.C, t.c);
  float g1[K1], x1[K1], g0[K0], x0[K0], uv[K0];
#pragma unroll
  for (int k = 0; k < K1; ++k) {
    const int l = l0 - HALO + run + RUNS * k;
    g1[k] = load(dy1, l);
    x1[k] = load(pre1, l);
  }
#pragma unroll
  for (int k = 0; k < K0; ++k) {
    const int l = l0 - HALO / 2 + run * K0 + k;
    g0[k] = load(dy0, l);
    x0[k] = load(pre0, l);
    uv[k] = load(u, l);
  }
#pragma unroll
  for (int k = 0; k < K1; ++k) {
    const int j = run + RUNS * k;
    const float sg = sigmoidf_(x1[k]);
    d1[j][cl] = g1[k] * (sg * (1.0f + x1[k] * (1.0f - sg)));   // (zero outside the sequence, as y0 and u)
  }
  float sg0[K0];
#pragma unroll
  for (int k = 0; k < K0; ++k) {
    const int j = run * K0 + k;
    sg0[k] = sigmoidf_(x0[k]);
    dw_st<BF>(&y0[0][0], j * CH + cl, x0[k] * sg0[k]);   // the second convolution's input
    dw_st<BF>(&us[0][0], j * CH + cl, uv[k]);
  }
  __syncthreads();
  {
    float v[K0 + HALO];
#pragma unroll
    for (int k = 0; k < K0 + HALO; ++k) v[k] = d1[run * K0 + k][cl];
#pragma unroll
    for (int k = 0; k < K0; ++k) {
      const int j = run * K0 + k;
      float g = g0[k];
      // y0[l] feeds pre1[l + 3 - i] through tap i
#pragma unroll
      for (int i = 0; i < DW_TAPS; ++i) g = fmaf(w[1][i], v[k + HALO - i], g);
      g = in(l0 - HALO / 2 + j) ? g * sg0[k] * (1.0f + x0[k] * (1.0f - sg0[k])) : 0.0f;
      d0[j][cl] = g;
    }
  }
  __syncthreads();
  const DwRows<BF> du_rows(FAR ? nullptr : dw_at<IO>(p.du, (long)t.b * p.du_bs), p.du_ls, p.C, l0, min(l0 + T, p.L), t.c, t.have);
  float gw[2][DW_TAPS + 1];   // taps, bias
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j <= DW_TAPS; ++j) gw[s][j] = 0.0f;
  {
    float v0[K + HALO], yv[K + HALO], u_[K + HALO];
#pragma unroll
    for (int k = 0; k < K + HALO; ++k) {
      const int j = run * K + k;
      v0[k] = d0[j][cl];
      yv[k] = dw_ld<BF>(&y0[0][0], j * CH + cl);
      u_[k] = dw_ld<BF>(&us[0][0], j * CH + cl);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int l = l0 + run * K + k;
      float du = 0.0f;
#pragma unroll
      for (int i = 0; i < DW_TAPS; ++i) du = fmaf(w[0][i], v0[k + HALO - i], du);
      const float e0 = v0[k + HALO / 2], e1 = d1[run * K + k + HALO][cl];   // dpre[0][l], dpre[1][l]: zero behind the end
#pragma unroll
      for (int i = 0; i < DW_TAPS; ++i) {
        gw[0][i] = fmaf(e0, u_[k + i], gw[0][i]);
        gw[1][i] = fmaf(e1, yv[k + i], gw[1][i]);
      }
      gw[0][DW_TAPS] += e0;
      gw[1][DW_TAPS] += e1;
      if constexpr (FAR) {
        if (p.du && t.have && l < p.L) dw_st<BF>(p.du, (long)t.b * p.du_bs + (long)l * p.du_ls + t.c, du);
      } else {
        du_rows.store(l - l0, du);
      }
    }
  }
  // a wave's two runs, then the four waves
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j <= DW_TAPS; ++j) {
      const float v = gw[s][j] + __shfl_xor(gw[s][j], 32, 64);
      if (!(run & 1)) red[(run >> 1) * 16 + s * 8 + j][cl] = v;
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 16 / RUNS; ++q) {
    const int sj = run + RUNS * q;
    if (t.have) p.partial[((long)t.row * 16 + sj) * p.C + t.c] = (red[sj][cl] + red[16 + sj][cl]) + (red[32 + sj][cl] + red[48 + sj][cl]);
  }
}

// dw[s][c][j], dbias[s][c] = fixed-order sums over the partial rows: workgroup = 32 columns x 8 row groups
__global__ __launch_bounds__(NTHREADS) void k_dwconv_dw(DwConvP p) {
  __shared__ float red[NTHREADS];
  const int ncol = p.nsets * 8 * p.C;  // column = (s * 8 + j) * C + c
  const int col = blockIdx.x * 32 + (threadIdx.x & 31), g = threadIdx.x >> 5;
  float a0 = 0.0f, a1 = 0.0f;
  if (col < ncol) {
    int r = g;
    // latency: the adds are a chain in a fixed order, but the loads of eight rounds travel together (12.2 -> 5.1 us at 8 x 1024
    // tokens, 290 channels)
#pragma unroll 8
    for (; r + 8 < p.nrows; r += 16) {
      a0 += p.partial[(long)r * ncol + col];
      a1 += p.partial[(long)(r + 8) * ncol + col];
    }
    if (r < p.nrows) a0 += p.partial[(long)r * ncol + col];
  }
  red[threadIdx.x] = a0 + a1;
  __syncthreads();
  if (g == 0 && col < ncol) {
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) t += red[i * 32 + (threadIdx.x & 31)];
    const int c = col % p.C, sj = col / p.C, s = sj >> 3, j = sj & 7;
    if (j < DW_TAPS) p.dw[((long)s * p.C + c) * DW_TAPS + j] = t;
    else p.dbias[(long)s * p.C + c] = t;
  }
}

int dwconv_partial_rows(int B, int L, bool chain) {
  const int tokens = chain ? DW_CHAIN_BWD : DW_BWD;
  return B * ((L + tokens - 1) / tokens);
}

static long dw_items(const DwConvP& p, int tokens) { return (long)p.B * ((p.L + tokens - 1) / tokens) * p.C; }
static unsigned dw_blocks(const DwConvP& p, int tokens) { return (unsigned)((dw_items(p, tokens) + NTHREADS - 1) / NTHREADS); }

template <int TL>
static int launch_dwconv_fwd_t(const DwConvP& p, hipStream_t st) {
  const dim3 g(dw_blocks(p, TL)), b(NTHREADS);
  if (p.dtype) {
    if (p.nsets == 1) hipLaunchKernelGGL((k_dwconv_fwd<true, 1, TL>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_dwconv_fwd<true, 2, TL>), g, b, 0, st, p);
  } else {
    if (p.nsets == 1) hipLaunchKernelGGL((k_dwconv_fwd<false, 1, TL>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_dwconv_fwd<false, 2, TL>), g, b, 0, st, p);
  }
  return (int)hipGetLastError();
}
int launch_dwconv_fwd(const DwConvP& p, hipStream_t st) {
  if (p.chain) {
    auto go = [&](auto kern, unsigned blocks) { hipLaunchKernelGGL(kern, dim3(blocks), dim3(NTHREADS), 0, st, p); };
    // Past what the last cache holds (256 MB of u, y and pre), the pieces of lines that tiles side by side write reach memory: in fp32 a thread's
    // channel, whose wave writes 256 bytes of a row, is ahead again, in bf16 tiles of 128 tokens (buffers in turn, us, threads of 16 tokens, tiles of 64 and of 128:
    // fp32 24 x 2048 tokens, 290 channels 86, 94, 101; 16 x 4096 113, 125, 137; 16 x 2048, 514 95, 105, 96; 1026 183, 214, 234; and below, 16 x 2048, 290 59, 58, 57;
    // 16 x 1000, 514 50, 45, 46; bf16 16 x 2048, 1026 120, 132, 112; 32 x 4096, 288 133, 123, 100; 16 x 4096, 290 74, 75, 65).
    const bool beyond = 5.0 * p.B * p.L * p.C * (p.dtype ? 2 : 4) > (double)(256 << 20);
    if (!dw_near(p)) p.dtype ? go(&k_dwconv_chain_fwd_threads<true, 4>, dw_blocks(p, 4)) : go(&k_dwconv_chain_fwd_threads<false, 4>, dw_blocks(p, 4));
    else if (beyond) p.dtype ? go(&k_dwconv_chain_fwd<true, 128>, dw_tiles(p, 128)) : go(&k_dwconv_chain_fwd_threads<false, 16>, dw_blocks(p, 16));
    else if (dw_tiles(p, 64) >= 1024) p.dtype ? go(&k_dwconv_chain_fwd<true, 64>, dw_tiles(p, 64)) : go(&k_dwconv_chain_fwd<false, 64>, dw_tiles(p, 64));
    else p.dtype ? go(&k_dwconv_chain_fwd<true, 16>, dw_tiles(p, 16)) : go(&k_dwconv_chain_fwd<false, 16>, dw_tiles(p, 16));
    return (int)hipGetLastError();
  }
  constexpr long waves = 2048 * 64;   // lanes of two waves a SIMD
  if (dw_items(p, 16) >= waves) return launch_dwconv_fwd_t<16>(p, st);
  if (dw_items(p, 8) >= waves) return launch_dwconv_fwd_t<8>(p, st);
  return launch_dwconv_fwd_t<4>(p, st);
}

int launch_dwconv_bwd(const DwConvP& p_, hipStream_t st) {
  DwConvP p = p_;
  p.nrows = dwconv_partial_rows(p.B, p.L, p.chain);
  const dim3 g(p.chain ? dw_tiles(p, DW_CHAIN_BWD) : dw_blocks(p, DW_BWD)), b(NTHREADS);
  if (p.chain) {
    const bool far = !dw_near(p);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, b, 0, st, p); };
    if (p.dtype) far ? go(&k_dwconv_chain_bwd<true, true>) : go(&k_dwconv_chain_bwd<true, false>);
    else far ? go(&k_dwconv_chain_bwd<false, true>) : go(&k_dwconv_chain_bwd<false, false>);
  } else if (p.dtype) {
    if (p.nsets == 1) hipLaunchKernelGGL((k_dwconv_bwd<true, 1>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_dwconv_bwd<true, 2>), g, b, 0, st, p);
  } else {
    if (p.nsets == 1) hipLaunchKernelGGL((k_dwconv_bwd<false, 1>), g, b, 0, st, p);
    else hipLaunchKernelGGL((k_dwconv_bwd<false, 2>), g, b, 0, st, p);
  }
  int e = (int)hipGetLastError();
  if (e || !p.dw) return e;
  hipLaunchKernelGGL(k_dwconv_dw, dim3((p.nsets * 8 * p.C + 31) / 32), b, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
