// Device-side building blocks shared by the ISSM kernels (gfx950 / CDNA4 only).
//
// Tiling conventions used by every kernel in this directory
//  * one workgroup = 256 threads = 4 wavefronts of 64 lanes;
//  * time is cut into chunks of CS = 64 tokens, the state dimension into slices of NS = 64
//    columns; a "unit" is one (batch*direction, chunk, head);
//  * every LDS tile is a row-major float array whose leading dimension is (width + 4): with
//    ld = 4 (mod 8) both fragment access patterns below are free of bank conflicts;
//  * matrix products run on v_mfma_f32_16x16x4_f32.  Lane (cm = lane & 15, g4 = lane >> 4)
//    feeds the j-th of four back-to-back MFMAs with k = kb + 4 g4 + j, so that an operand
//    stored with k contiguous ("M-major", tile[m][k]) is fetched with one 128-bit LDS read and
//    an operand stored with m contiguous ("K-major", tile[k][m]) with four 32-bit reads.  The
//    accumulator register r of that lane holds element (row = 4 g4 + r, col = cm) of the
//    16x16 result;
//  * "column-lane layout": a wave owns 16 state columns, lane (cm, g4) owns column cm and the
//    16 chunk rows {16J + 4 g4 + j : J, j = 0..3}, array index k = 4J + j.  A lane then holds
//    exactly the elements it feeds as the K-major B operand of a product that contracts over
//    rows, and exactly the accumulator rows it gets back from a product whose output rows are
//    chunk rows, so cumulative sums, decays and all elementwise work stay in registers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

// A wave-uniform value made opaque to the optimizer (its multiples are then formed next to their use instead of being
// hoisted out of loops into scarce scalar registers).  A translation unit may define its own form before including this.
#ifndef ISSM_OPAQUE_S
#define ISSM_OPAQUE_S(x) asm volatile("" : "+s"(x))
#endif

namespace issm {

constexpr int CS = 64;         // tokens per chunk
constexpr int NS = 64;         // state columns per slice
constexpr int LDN = NS + 4;    // leading dimension of [*][NS] tiles
constexpr int LDC = CS + 4;    // leading dimension of [*][CS] tiles
constexpr int MAXP = 64;       // largest head dimension built
constexpr int NTHREADS = 256;
constexpr int NCU = 256;       // compute units of the card
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

// Whether k_chunk_scan and k_bwd_dx take two groups of four waves a workgroup, each with every second slice of the states: where no CU
// gets a second workgroup.  A lone wave on a SIMD issues a vector instruction every 5.3 cycles, two together every 2.7 to 4.5.  256 units
// of four slices: k_chunk_scan 13.2 -> 11.4 us (fp32, heads of 32), 14.3 -> 10.8 (bf16, 36), k_bwd_dx 15.6 -> 12.7 (128 units) and 17.4 ->
// 13.9; 512 units, which share the CUs either way: 16.5 with one group, 18.8 with two.  (k_local_tile, bound by issue in its steps, the same
// way: 17.6 -> 17.4 us, bf16 without a gradient 22.7 -> 23.9.)
inline bool two_groups(int units, int N) { return units <= NCU && N > NS; }

typedef float f4 __attribute__((ext_vector_type(4)));

struct TensorD {
  const void* ptr;
  long s0, s1, s2;  // element strides of dims 0,1,2 (innermost contiguous)
};

// Division of a number below 2^31 by a fixed one in four instructions: m = (2^32 - 1) / d, the quotient one short at most.
struct Div {
  unsigned d, m;
  // n becomes the quotient; returns the remainder
  __device__ __forceinline__ unsigned operator()(unsigned& n) const {
    unsigned q = __umulhi(n, m), r = n - q * d;
    const bool more = r >= d;
    q += more ? 1u : 0u;
    r -= more ? d : 0u;
    n = q;
    return r;
  }
};
static inline Div div_by(unsigned d) { return Div{d, 0xffffffffu / d}; }

// Kernel parameter block (passed by value).  What a kernel needs before its first request -- sizes and divisors to find its unit, the inputs'
// addresses -- lies in front, in few cache lines.
struct KP {
  int B, L, H, P, N, G, ndir, nc, hpg;
  int dir0;  // direction handled by this launch (kernels launched per direction)
  int io_dt, dt_dt, h0_dt;  // 0 = f32, 1 = bf16
  unsigned flags;
  float dt_min, dt_max;
  // full_tiles picks the kernel variants: 1 = every chunk has 64 rows and every column slice 64 columns (complete-tile code); 0 = the
  // "edge" variants (FULL = false), the same code with clamped addresses, dt' = 0 where a row or column is absent and
  // guarded stores in the workgroups and steps that have such rows or columns.
  int full_tiles;
  Div by_H, by_nc, by_hpg, by_slices, by_G, by_quads, by_P;   // slices, quads: of 64 and 4 state columns
  TensorD x[2], Bm[2], Cm[2], z[2], out[2], dout[2], dx[2], dB[2], dC[2], dz[2];
  TensorD dt, ddt, h0;
  // Two directions with a bf16 ddt: the first direction's share of ddt travels in fp32 through this (B, L, H, N) buffer
  // instead of through ddt itself, so that the sum of the two is rounded to bf16 once (null: it travels through ddt).
  TensorD ddt_part;
  // bf16 inputs, incomplete tiles: sums of dB and dC over the heads the tile-base chunk backward evaluated, in fp32, of the
  // workgroups with heads it left to the level form (which goes on from them, so that dB and dC are rounded once, as where
  // the level form evaluates all heads): per direction and workgroup the lanes' 16 + 16 values [32][NTHREADS].  Null: they
  // travel through dB and dC themselves.  (Complete tiles do that: six decoder layers, a training step, 7.38 against 7.52 ms.)
  // Where several workgroups of the tile-base kernel share the heads of a group (bwd_head_parts), the sums of all workgroups in
  // all cases, one such array per part, which k_bwd_parts_sum adds up.
  float* dbc_part;
  const float* A;
  const float* D;
  const float* dt_bias;
  float* final_states[2];
  const float* dfinal[2];
  const int* seq_idx;   // (B, L) sequence ids of packed rows, or null
  long seq_s0, seq_s1;
};

enum : unsigned { F_SOFTPLUS = 1u, F_D_HDIM = 2u, F_NOCLAMP = 4u };
// What the running sum of dt' A log2(e) takes where the sequence id changes: decays across the change become 2^-128.
constexpr float SEQ_CUT = 128.0f;

// Parameter block of the gated RMSNorm kernels.
struct NormP {
  long rows;
  int ncols, gs, ngroups;
  int dt, wdt, nbg;
  float eps;
  const void *x, *z, *w;
  long xs, zs;
  void* y;
  long ys;
  float* rstd;
  const void* dy;
  long dys;
  void *dx, *dz;
  long dxs, dzs;
  float* dw_partial;
  void* dw;         // (ncols) of dw_dt, as db
  int dw_dt;
  int nblocks;
  int ln;           // LayerNorm statistics (mean subtracted) instead of RMS
  const void* b;    // bias in the weight's dtype, or null
  float* mean;
  float* db_partial;
  void* db;
};

// parameters of the serialization-code kernel (hilbert.hip)
struct HilbertP {
  int B, N, bits;
  int perm[3];          // grid coordinate used as first / second / third curve coordinate
  float cell;
  const float* points;  // (B, N, 3)
  const float* mins;    // (B, 3) per-sample minimum corner
  long* codes;          // (B, N)
};

// the whole serialization in one launch (hilbert.hip): index / inverse (norder, B, N), NP = N rounded up to a power of two
struct HilbertOrderP {
  int B, N, NP, bits, norder;
  int perm[6][3];
  float cell;
  const float* points;
  long* index;
  long* inverse;  // may be null
};

// parameters of the encoding's table (box_dist.hip)
struct BoxTableP {
  int nodes, hidden, dtype, coords_dtype;
  const void *coords, *w1, *b1, *w2;
  float* table;
};
// parameters of the box-to-point distance encoding kernels (box_dist.hip)
struct BoxDistP {
  int B, L, K, D, H, W, dtype, nwg, nwg_bwd;
  const float* key;      // (B, L, 3)
  const float* corners;  // (B, K, 8, 3), or NULL with boxes given
  const float* boxes;    // (B, K, 7) centre, size, heading: corners (and the weight's centre / radius) derived from it
  float min_radius;
  const float* angle;    // (B, K) or NULL (zero)
  const float* table;    // (16, D, H, W)
  float log_scale, max_value;
  void* dist;            // (B, L, K, 16) io dtype, or NULL
  const float* qcenter;  // (B, K, 3), with radius (B, K): inputs of the locality weight
  const float* radius;
  float weight_dist;
  float* weights;        // (B, L, K) fp32, or NULL
  const void* ddist;     // (B, L, K, 16) io dtype
  void* partial;         // 2 words (scale) + (nwg_bwd, D*H*W, 16) 64-bit fixed-point words
  float* dtable;         // (16, D, H, W) fp32
};

// parameters of the depthwise conv + SiLU kernels (dwconv_silu.hip)
struct DwConvP {
  int B, L, C, nsets, dtype;
  int chain;           // nsets == 2: set 1 convolves set 0's output instead of u
  const void* u;       // (B, L, C) io dtype, element strides u_bs (batch), u_ls (token), channels contiguous
  long u_bs, u_ls;
  const float* w;      // (nsets, C, 7) fp32
  const float* bias;   // (nsets, C) fp32
  void* y;             // (nsets, B, L, C) io dtype; with split > 0: (nsets, B, L, split), channels [0, split)
  void* y_tail;        // split > 0: (nsets, B, L, C - split), channels [split, C)
  int split;
  void* pre;           // (nsets, B, L, C) io dtype: convolution output before SiLU (saved for the backward)
  const void* dy[2];   // (B, L, C) io dtype per set, or NULL; with split > 0: (B, L, split)
  const void* dy_tail[2];  // split > 0: (B, L, C - split) per set, or NULL
  void* du;            // (B, L, C) io dtype, element strides du_bs, du_ls, channels contiguous
  long du_bs, du_ls;
  float* partial;      // (nrows, nsets, 8, C) fp32
  int nrows;
  float* dw;           // (nsets, C, 7) fp32
  float* dbias;        // (nsets, C) fp32
};

// parameters of the kernels of transpose_states.hip
struct TrP {
  int B, R, C, in_dt, out_dt;
  const void* in0;
  const void* in1;
  void* out;
  float alpha;
};
struct LayerGradsP {
  const float *conv, *gen, *gen_bias, *norm;   // (conv_rows, 2, 8, C), (gen_rows, R0, 16), (gen_rows, R0), (norm_rows, di)
  int conv_rows, gen_rows, norm_rows;
  int C, H, R0, di, K, nD;
  const float *dA, *A, *dD;                    // (H, K), (H, K), (nD)
  void* out;
  int bf16;
  int b_gen, b_bias, b_norm, b_A, b_D, b_tr;   // first workgroup of each kind
};

// parameters of the dt / B / C generation kernels (param_gen.hip)
// parameters of the layer-parameter kernel (layer_params.hip)
constexpr int LAYER_ARRAYS = 9;
struct LinearJob {
  const uint16_t *x, *w;
  uint16_t* y;
  int tokens, out, steps, oblocks;   // steps of 32 along the contraction
  int turn;                          // 0: y (tokens, out); else y (tokens / turn, out, turn)
};
struct LinearP {
  LinearJob job[2];
  int blocks0, blocks1;   // of the first, of both
};
// parameters of the products of many tokens (linear_tile.hip)
struct LinearTileJob {
  const uint16_t *x, *w;
  uint16_t* y;
  int tokens, in, out, otiles;
};
struct LinearTileP {
  LinearTileJob job[2];
  int blocks0;
};
// parameters of the projections' weight gradient (linear_dw.hip)
struct LinearDwP {
  const uint16_t *dy, *x;   // (tokens, out), (tokens, in)
  float* partial;           // (splits, out, in)
  uint16_t* dw;             // (out, in)
  int tokens, in, out, splits, btiles, per;
};
struct LinearDwJobs {
  LinearDwP job[2];
  int blocks0, sums0;       // workgroups of the first, of its sums
};
// parameters of the kernel behind the scan (layer_out.hip)
struct LayerOutP {
  const uint16_t *y0, *y1, *z, *kw, *qw, *qb;   // qw, qb may be NULL
  uint16_t *key, *query;
  const float *last0, *last1;
  long rows, zs;   // rows of y, row stride of z
  int B, K, di, key_blocks;
  float keps, qeps;
};
struct LayerParamsP {
  const void* src[LAYER_ARRAYS];
  int n[LAYER_ARRAYS], bf16[LAYER_ARRAYS];
  int total, a_log, H, K;   // sum of n; which array is A_log
  float* out;               // (total)
  float* A;                 // (H, K)
};

struct PGenP {
  long tokens;
  int K, H, G, dtype, has_back;
  const void* dist;      // (tokens, K, M) io dtype
  const float* W;        // (R0, M) fp32
  const float* bias;     // (tokens, R) fp32, R = R0 + (has_back ? 2G : 0), or NULL with the three below:
  const void* tok;       // io dtype, row of H values per token, tok_stride elements apart
  long tok_stride;
  const float* tok_add;  // (H)
  const void* tail;      // (has_back ? 2 : 1, tokens, 2G) io dtype
  void *dt, *Bm, *Cm, *Bb, *Cb;                    // (tokens, H|G, K) io dtype
  const float* weights;  // (tokens, K) fp32 or NULL: dt = softplus(raw) * weights instead of raw
  void* dt_raw;          // (tokens, H, K) io dtype: raw dt, written by the forward when weights is given
  float* dweights;       // (tokens, K) fp32 or NULL
  const void *ddt, *dB, *dC, *dBb, *dCb;           // gradients of the outputs
  void* ddist;           // (tokens, K, M) io dtype
  float* dbias;          // (tokens, R) fp32
  float* dbias_sum;      // (R) fp32 or NULL: dbias summed over the tokens
  float* dw_partial;     // (nblocks, R0, M) fp32
  float* dW;             // (R0, M) fp32 or NULL: dw_partial is what the caller wants, and
  void *dtok, *dtail;    // the bias gradients in io dtype, (tokens, H) rows dtok_stride apart, (2, tokens, 2G), or NULL,
  long dtok_stride;
  float* bias_partial;   // and the first R0 summed over a workgroup's tokens, (nblocks, R0)
  int nblocks;
};

// two floats -> two bf16 (round to nearest even) in one dword
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float fl2 __attribute__((ext_vector_type(2)));
  const bf2 h = __builtin_convertvector((fl2){lo, hi}, bf2);
  return __builtin_bit_cast(unsigned, h);
}

__device__ __forceinline__ float bf16_to_f(uint16_t v) { return __uint_as_float(((uint32_t)v) << 16); }
// round to nearest even; the hardware conversion (v_cvt_pk_bf16_f32), one instruction per two values
__device__ __forceinline__ uint16_t f_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
// a float rounded to bf16 (nearest even) and back
__device__ __forceinline__ float bf16_round(float f) { return (float)(__bf16)f; }
// runtime-dtype element access (used only outside hot loops)
__device__ __forceinline__ float ldv(const void* p, long i, int dt) {
  return dt ? bf16_to_f(((const uint16_t*)p)[i]) : ((const float*)p)[i];
}
__device__ __forceinline__ void stv(void* p, long i, int dt, float v) {
  if (dt) ((uint16_t*)p)[i] = f_to_bf16(v); else ((float*)p)[i] = v;
}
__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }
// (the hardware exp2 / log2 directly: the arguments here need none of the library's range fix-ups --
// 1 + exp(x) >= 1 is never denormal and an exp that underflows to 0 is the right answer)
__device__ __forceinline__ float sigmoidf_(float x) { return __builtin_amdgcn_rcpf(1.0f + ex2(-x * LOG2E)); }
// softplus as the reference evaluates it: log(exp(x) + 1) for x <= 20, identity above
__device__ __forceinline__ float softplus_(float x) {
  return x <= 20.0f ? LN2 * __builtin_amdgcn_logf(1.0f + ex2(x * LOG2E)) : x;
}

// Batched global loads / stores of one element type: all CNT accesses are issued before any
// value is consumed.  The address is (uniform element offset ubase) + (per-lane 32-bit element
// offset off[i]), which lets the compiler keep the base in scalar registers; off[i] < 0 marks an
// absent element (load: reads as 0, the access itself goes to offset 0; store: skipped).
template <bool BF, int CNT>
__device__ __forceinline__ void gload(const void* p, long ubase, const int (&off)[CNT], float (&out)[CNT]) {
  if (BF) {
    const uint16_t* q = (const uint16_t*)p + ubase;
    uint16_t r[CNT];
#pragma unroll
    for (int i = 0; i < CNT; ++i) r[i] = q[off[i] < 0 ? 0 : off[i]];
#pragma unroll
    for (int i = 0; i < CNT; ++i) out[i] = off[i] < 0 ? 0.0f : bf16_to_f(r[i]);
  } else {
    const float* q = (const float*)p + ubase;
    float r[CNT];
#pragma unroll
    for (int i = 0; i < CNT; ++i) r[i] = q[off[i] < 0 ? 0 : off[i]];
#pragma unroll
    for (int i = 0; i < CNT; ++i) out[i] = off[i] < 0 ? 0.0f : r[i];
  }
}
template <bool BF, int CNT>
__device__ __forceinline__ void gstore(void* p, long ubase, const int (&off)[CNT], const float (&v)[CNT]) {
  if (BF) {
    uint16_t* q = (uint16_t*)p + ubase;
#pragma unroll
    for (int i = 0; i < CNT; ++i)
      if (off[i] >= 0) q[off[i]] = f_to_bf16(v[i]);
  } else {
    float* q = (float*)p + ubase;
#pragma unroll
    for (int i = 0; i < CNT; ++i)
      if (off[i] >= 0) q[off[i]] = v[i];
  }
}

// Opaque pass-through of registers: everything that depends on the values is ordered after this
// point and everything that produces them before, which keeps the phases of a long straight-line
// kernel from being interleaved by the scheduler (and their temporaries from being live together).
__device__ __forceinline__ void pin16(float (&a)[16]) {
  asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]),
               "+v"(a[8]), "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15]));
}
__device__ __forceinline__ void pin4(f4& a) { asm volatile("" : "+v"(a)); }
// Workgroups are dealt round-robin to the 8 XCDs; give each XCD a contiguous range of logical
// ids so that units sharing B/C tiles (the heads of one chunk) share an L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
  if (nblocks & 7) return bid;
  return (bid & 7) * (nblocks >> 3) + (bid >> 3);
}

__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc += A(16 x 16k) * B(16k x 16) for k in [kb, kb+16); both operands M-major:
// A[m][k] at a[(m0+m)*lda + k], B[n][k] at b[(n0+n)*ldb + k].
__device__ __forceinline__ void mma16_mm(f4& acc, const float* a, int lda, int m0, const float* b, int ldb,
                                         int n0, int kb, int lane) {
  const int m = lane & 15, g = lane >> 4;
  f4 av = *(const f4*)(a + (m0 + m) * lda + kb + 4 * g);
  f4 bv = *(const f4*)(b + (n0 + m) * ldb + kb + 4 * g);
  acc = mfma4(av.x, bv.x, acc);
  acc = mfma4(av.y, bv.y, acc);
  acc = mfma4(av.z, bv.z, acc);
  acc = mfma4(av.w, bv.w, acc);
}
// both operands K-major: A[k][m] at a[k*lda + m0+m], B[k][n] at b[k*ldb + n0+n]
__device__ __forceinline__ void mma16_kk(f4& acc, const float* a, int lda, int m0, const float* b, int ldb,
                                         int n0, int kb, int lane) {
  const int m = lane & 15, g = lane >> 4;
  const float* ap = a + (kb + 4 * g) * lda + m0 + m;
  const float* bp = b + (kb + 4 * g) * ldb + n0 + m;
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = mfma4(ap[j * lda], bp[j * ldb], acc);
}
// A M-major, B K-major
__device__ __forceinline__ void mma16_mk(f4& acc, const float* a, int lda, int m0, const float* b, int ldb,
                                         int n0, int kb, int lane) {
  const int m = lane & 15, g = lane >> 4;
  f4 av = *(const f4*)(a + (m0 + m) * lda + kb + 4 * g);
  const float* bp = b + (kb + 4 * g) * ldb + n0 + m;
  acc = mfma4(av.x, bp[0], acc);
  acc = mfma4(av.y, bp[ldb], acc);
  acc = mfma4(av.z, bp[2 * ldb], acc);
  acc = mfma4(av.w, bp[3 * ldb], acc);
}

// ------------------------------------------------------------------ split-bf16 products
// v_mfma_f32_16x16x4_f32 shares the vector ALU's issue slots (measured: its time adds to the VALU time
// instead of overlapping it), while v_mfma_f32_16x16x32_bf16 does 8x the multiply-adds in about half the
// time.  Where both operands of a product are reused often enough to amortise the conversion, an fp32
// product a.b is therefore evaluated as  ah.bh + ah.bl + al.bh  with a = ah + al, ah = bf16(a),
// al = bf16(a - ah) (16 significand bits per operand; the dropped al.bl term is <= 2^-16 |a.b|) and fp32
// accumulation.  One instruction contracts over K = 32: lane (cm, g4) supplies k-slots 0..7 of group g4.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4 mfma_bf(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// acc += A.B with both operands given as (hi, lo) pairs
__device__ __forceinline__ f4 mfma_split(bf8 ah, bf8 al, bf8 bh, bf8 bl, f4 c) {
  c = mfma_bf(al, bh, c);
  c = mfma_bf(ah, bl, c);
  return mfma_bf(ah, bh, c);
}
// Two values at a time: each conversion instruction rounds a pair, and left to itself the compiler rounds every value once more,
// alone, for the subtraction (52 instructions of 860 in a step of k_local_tile with fp32 inputs, two head tiles).
__device__ __forceinline__ void split_pair(float a, float b, unsigned& hi, unsigned& lo) {
  hi = pack_bf16(a, b);
  lo = pack_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}
__device__ __forceinline__ void split4(const float (&v)[4], bf4& hi, bf4& lo) {
  uint2 h, l;
  split_pair(v[0], v[1], h.x, l.x);
  split_pair(v[2], v[3], h.y, l.y);
  hi = __builtin_bit_cast(bf4, h);
  lo = __builtin_bit_cast(bf4, l);
}
// eight fp32 values of a lane (k-slots 0..7) -> (hi, lo) fragments
__device__ __forceinline__ void split8(const float (&v)[8], bf8& hi, bf8& lo) {
  uint4 h, l;
  split_pair(v[0], v[1], h.x, l.x);
  split_pair(v[2], v[3], h.y, l.y);
  split_pair(v[4], v[5], h.z, l.z);
  split_pair(v[6], v[7], h.w, l.w);
  hi = __builtin_bit_cast(bf8, h);
  lo = __builtin_bit_cast(bf8, l);
}
// Row-major bf16 tiles [rows][SplitLd] holding the hi and the lo halves of an fp32 (rows x KW) tile, KW a
// multiple of 16.  Fragment of K-step t for lane (row, g4): columns 32t + 4 g4 .. +3 and 32t + 16 + 4 g4 .. +3,
// i.e. k-slot s <-> column 32t + 16 (s >> 2) + 4 g4 + (s & 3).
template <int KW>
struct SplitTile {
  static constexpr int LD = KW + 8;
  uint16_t hi[CS * LD];
  uint16_t lo[CS * LD];
};
// (HALF: the tile has no columns 32t + 16 .. 32t + 31; those k-slots read as zero.)
template <int LD, bool HALF = false>
__device__ __forceinline__ bf8 split_frag(const uint16_t* tile, int row, int g4, int t) {
  const uint16_t* q = tile + row * LD + 32 * t + 4 * g4;
  const bf4 a = *(const bf4*)q;
  bf4 b = {0, 0, 0, 0};
  if (!HALF) b = *(const bf4*)(q + 16);
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
// Store of a cooperative (64 x 16 PT) register tile (layout of lp_load) as split bf16 tiles.
template <int PT, int LD>
__device__ __forceinline__ void lp_store_split(const float (&v)[CS * PT * 16 / NTHREADS], uint16_t* hi, uint16_t* lo,
                                               int tid = threadIdx.x) {
  constexpr int G4 = 4 * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e4 = tid + i * NTHREADS, o = (e4 / G4) * LD + (e4 % G4) * 4;
    const float w[4] = {v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    bf4 h, l;
    split4(w, h, l);
    *(bf4*)(hi + o) = h;
    *(bf4*)(lo + o) = l;
  }
}

// Same register tile stored transposed, [p][l] (rows = head dimension, KW = CS columns), for products that
// contract over the rows of the chunk.
template <int PT, int LD, bool SPLIT = true>
__device__ __forceinline__ void lp_store_split_t(const float (&v)[CS * PT * 16 / NTHREADS], uint16_t* hi,
                                                 uint16_t* lo, int tid = threadIdx.x) {
  constexpr int G4 = 4 * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      unsigned h, w;
      split_pair(v[4 * i + j], v[4 * i + j + 1], h, w);
      hi[(p4 + j) * LD + l] = (uint16_t)h;
      hi[(p4 + j + 1) * LD + l] = (uint16_t)(h >> 16);
      if (SPLIT) {
        lo[(p4 + j) * LD + l] = (uint16_t)w;
        lo[(p4 + j + 1) * LD + l] = (uint16_t)(w >> 16);
      }
    }
  }
}
// acc[pt] += (tile^T)(16 pt .. +15, :) . b  for a product over the 64 chunk rows whose B operand is the lane's
// 16 column-lane values (k = 4J + j <-> row 16J + 4 g4 + j): two K = 32 steps, step t <-> values 8t .. 8t+7.
// `b(k)` yields the lane's value k (evaluated step by step, so that only eight are live at a time).
// MODE 1: both operands as (hi, lo) pairs, three instructions per step.  MODE 0: both operands rounded to bf16, one
// instruction.  MODE 2: the tile is exact in bf16 (bf16 inputs), only b is split: two instructions.
template <int PT, int LD, int MODE = 1, typename F>
__device__ __forceinline__ void rows_product_split(f4 (&acc)[PT], const uint16_t* thi, const uint16_t* tlo, F b,
                                                   int cm, int g4) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = b(8 * t + j);
    bf8 bh, bl;
    if (MODE != 0) {
      split8(w, bh, bl);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) bh[j] = (__bf16)w[j];
    }
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) {
      const bf8 ah = split_frag<LD>(thi, pt * 16 + cm, g4, t);
      if (MODE == 1) {
        const bf8 al = split_frag<LD>(tlo, pt * 16 + cm, g4, t);
        acc[pt] = mfma_split(ah, al, bh, bl, acc[pt]);
      } else if (MODE == 2) {
        acc[pt] = mfma_bf(ah, bl, acc[pt]);
        acc[pt] = mfma_bf(ah, bh, acc[pt]);
      } else {
        acc[pt] = mfma_bf(ah, bh, acc[pt]);
      }
    }
  }
}

// a (64 x 16 PT) register tile (layout of lp_load) as bf16 into LDS dst[l][p]
template <int PT, int LD>
__device__ __forceinline__ void lp_store_bf(const float (&v)[CS * PT * 16 / NTHREADS], uint16_t* dst, int tid) {
  constexpr int G4 = 4 * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e4 = tid + i * NTHREADS;
    *(uint2*)(dst + (e4 / G4) * LD + (e4 % G4) * 4) =
        make_uint2(pack_bf16(v[4 * i], v[4 * i + 1]), pack_bf16(v[4 * i + 2], v[4 * i + 3]));
  }
}

// The same (see warm_args) for a kernel whose first BYTES bytes of arguments are other blocks.
template <int BYTES>
__device__ __forceinline__ void warm_first() {
  static_assert(BYTES > 3 * 64 && BYTES <= 9 * 64, "four to nine lines");
  unsigned t;
  const auto args = __builtin_amdgcn_kernarg_segment_ptr();
#define ISSM_WARM_4 "s_load_dword %0, %1, 0x0\ns_load_dword %0, %1, 0x40\ns_load_dword %0, %1, 0x80\ns_load_dword %0, %1, 0xc0\n"
#define ISSM_WARM(lines_) asm volatile(ISSM_WARM_4 lines_ "s_waitcnt lgkmcnt(0)" : "=&s"(t) : "s"(args))
#define ISSM_WARM_AT(at_) "s_load_dword %0, %1, " at_ "\n"
  if constexpr (BYTES <= 4 * 64) ISSM_WARM("");
  else if constexpr (BYTES <= 5 * 64) ISSM_WARM(ISSM_WARM_AT("0x100"));
  else if constexpr (BYTES <= 6 * 64) ISSM_WARM(ISSM_WARM_AT("0x100") ISSM_WARM_AT("0x140"));
  else if constexpr (BYTES <= 7 * 64) ISSM_WARM(ISSM_WARM_AT("0x100") ISSM_WARM_AT("0x140") ISSM_WARM_AT("0x180"));
  else if constexpr (BYTES <= 8 * 64) ISSM_WARM(ISSM_WARM_AT("0x100") ISSM_WARM_AT("0x140") ISSM_WARM_AT("0x180") ISSM_WARM_AT("0x1c0"));
  else ISSM_WARM(ISSM_WARM_AT("0x100") ISSM_WARM_AT("0x140") ISSM_WARM_AT("0x180") ISSM_WARM_AT("0x1c0") ISSM_WARM_AT("0x200"));
#undef ISSM_WARM_AT
#undef ISSM_WARM
#undef ISSM_WARM_4
}

// Every line of a kernel's KP into the scalar cache at once.  Left to itself a kernel waits for one part of it after the other, six or
// seven times in front of its first request, and on a CU that has not run it just before each wait is a trip to the L2.  2 x 1024
// tokens, 8 heads x 32, 256 states, forward, one workgroup a CU: k_local_tile 18.4 -> 17.6 us, k_chunk_scan 13.5 -> 13.2, k_state_pass 6.9 -> 6.5;
// 2 x 160 tokens, 4 heads, training, sum of the kernels 88 -> 86; no difference with many workgroups a CU.
__device__ __forceinline__ void warm_args() {
  static_assert(sizeof(KP) >= 15 * 64 + 4, "the block is the kernel's first argument");
  unsigned t;
  asm volatile("s_load_dword %0, %1, 0x0\n"
               "s_load_dword %0, %1, 0x40\n"
               "s_load_dword %0, %1, 0x80\n"
               "s_load_dword %0, %1, 0xc0\n"
               "s_load_dword %0, %1, 0x100\n"
               "s_load_dword %0, %1, 0x140\n"
               "s_load_dword %0, %1, 0x180\n"
               "s_load_dword %0, %1, 0x1c0\n"
               "s_load_dword %0, %1, 0x200\n"
               "s_load_dword %0, %1, 0x240\n"
               "s_load_dword %0, %1, 0x280\n"
               "s_load_dword %0, %1, 0x2c0\n"
               "s_load_dword %0, %1, 0x300\n"
               "s_load_dword %0, %1, 0x340\n"
               "s_load_dword %0, %1, 0x380\n"
               "s_load_dword %0, %1, 0x3c0\n"
               "s_waitcnt lgkmcnt(0)" : "=&s"(t) : "s"(__builtin_amdgcn_kernarg_segment_ptr()));
}

// Decode a unit id -> (b, dir, c, h); h is fastest so that the heads of one chunk run back to
// back and share the B/C tiles in cache.
struct Unit {
  int b, dir, bt, c, h, g;
};
// Order of the units: heads fastest.  With two directions the next index is the direction, and chunk j of the
// forward direction is paired with chunk nc - 1 - j of the reversed one: the same block of tokens, so the two
// workgroups that read one head's dt tile (the largest operand, shared by the directions) run side by side on one
// XCD and the second read is served by its L2.
// Bound by the latency of what it does, in front of everything: with divisions and a branch on ndir 1300 - 2000 cycles of the 8700
// until k_local_tile's first step began, one workgroup a CU.
__device__ __forceinline__ Unit decode_unit(const KP& p, unsigned u) {
  Unit r;
  r.h = (int)p.by_H(u);
  const unsigned two = (unsigned)p.ndir - 1;
  r.dir = (int)(u & two);
  u >>= two;
  const int j = (int)p.by_nc(u);
  r.b = (int)u;
  r.c = r.dir ? p.nc - 1 - j : j;
  r.bt = r.b * p.ndir + r.dir;
  unsigned g = (unsigned)r.h;
  p.by_hpg(g);
  r.g = (int)g;
  return r;
}
// physical row of logical time t for a direction
__device__ __forceinline__ int phys_row(const KP& p, int dir, int t) { return dir ? p.L - 1 - t : t; }

// ---------------------------------------------------------------- column-lane layout helpers
// chunk row of array index k for lane group g4
__device__ __forceinline__ int lane_row(int k, int g4) { return 16 * (k >> 2) + 4 * g4 + (k & 3); }

// One value per lane group: the sums of the groups before and after the lane's own, and of all four, without LDS
// (v_permlane16_swap and v_permlane32_swap of a value with its own copy leave the even / odd rows of 16 lanes, the lower /
// upper half, on both).  The chunk backward's running and suffix sums: six trips through LDS a head fewer, fp32, both directions,
// 8 x 1024 tokens, 8 heads x 32, 256 states 205 -> 196 us; 4 x 1000, 36, 200 states 56.9 -> 55.4.  bf16 inputs (151 us either way) and
// the kernels that call lane_prep or take single sums gained nothing by it and keep the LDS form and its rounding.
__device__ __forceinline__ void group_sums(float c, int g4, float& before, float& after, float& all) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(c), __float_as_uint(c), false, false);
  const float even = __uint_as_float(r[0]), odd = __uint_as_float(r[1]), pair = even + odd;
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(pair), __float_as_uint(pair), false, false);
  const float lower = __uint_as_float(q[0]), upper = __uint_as_float(q[1]);
  all = lower + upper;
  before = (g4 & 1 ? even : 0.0f) + (g4 & 2 ? lower : 0.0f);
  after = (g4 & 1 ? 0.0f : odd) + (g4 & 2 ? 0.0f : upper);
}


// inclusive prefix / suffix over the four lane groups g4 = 0..3 (lanes cm, cm+16, cm+32, cm+48)
__device__ __forceinline__ float scan_g_incl(float v, int g4) {
  float t = __shfl_up(v, 16, 64);
  if (g4 >= 1) v += t;
  t = __shfl_up(v, 32, 64);
  if (g4 >= 2) v += t;
  return v;
}
__device__ __forceinline__ float scan_g_incl_rev(float v, int g4) {
  float t = __shfl_down(v, 16, 64);
  if (g4 <= 2) v += t;
  t = __shfl_down(v, 32, 64);
  if (g4 <= 1) v += t;
  return v;
}

// Where the lane's 16 chunk rows live in memory.  Element k = 4J + j is chunk row 16J + 4 g4 + j,
// i.e. physical row base + step * (16J + j): a per-lane part (base) plus a part that is the same
// for the whole wave, so that in a full chunk the address of every element is a scalar base
// plus ONE per-lane offset.  `full` (a compile-time constant of the kernel variant) says that all 64
// rows and all 64 columns of every slice exist (the head dimension is checked separately at run time).  Otherwise
// `edge` (uniform) says whether this chunk has fewer than 64 rows or the slice fewer than 64 columns: absent rows read
// zero and absent columns column 0 -- finite whenever the inputs are -- and everything that would let them act is zero:
// dt' (hence B dt' and the decays), x and dy rows, stored results.
struct RowMap {
  int base, step, nvalid, rows, cols;
  bool full, edge;
  unsigned long long cut;  // bit r: the sequence id changes between rows r - 1 and r of the chunk (scan order; the initial states count as id 0); uniform
};
template <bool FULL>
__device__ __forceinline__ RowMap make_rowmap(const KP& p, const Unit& u, int g4, int n0) {
  RowMap r;
  const int t0 = u.c * CS + 4 * g4;
  r.base = u.dir ? p.L - 1 - t0 : t0;
  r.step = u.dir ? -1 : 1;
  r.nvalid = min(CS, p.L - u.c * CS);
  // FULL kernels are only launched when every chunk and every column slice is complete
  r.full = FULL;
  r.rows = p.L;
  r.cols = p.N;
  r.edge = !FULL && (r.nvalid < CS || n0 + NS > p.N);
  r.cut = 0;
  if (!FULL && p.seq_idx) {  // packed sequences take the kernels' general variants
    // lane = row of the chunk in scan order; its predecessor in scan order may be the previous chunk's last row
    const int row = u.c * CS + (int)(threadIdx.x & 63);
    // The initial states belong to sequence id 0 (issm_chunk_scan.py:123 and issm_state_passing.py:91 start from id 0):
    // a row whose first id is not 0 is cut off from them, like a row from a predecessor of another id.
    bool changes = false;
    if (row < p.L) {
      const long t = u.dir ? p.L - 1 - row : row, tp = u.dir ? t + 1 : t - 1;
      const int* q = p.seq_idx + (long)u.b * p.seq_s0;
      changes = q[t * p.seq_s1] != (row > 0 ? q[tp * p.seq_s1] : 0);
    }
    r.cut = __ballot(changes);
  }
  return r;
}
// A (b, third) slab of a (B,L,G|H,N)-shaped tensor as a raw buffer: a load whose byte offset lies at or beyond the end
// of the slab's last row returns zero.  That covers the rows a chunk does not have at no cost
// per access: forwards they lie past the last row; backwards they lie before the first one, and a negative 32-bit offset
// is a very large one.  (The host keeps a slab below 2^32 bytes; within 63 rows of that an absent row's offset may wrap to
// one of another row: still inside the slab, and the value is not used.)  Word 3: raw 32-bit data format.
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slab_of(const T* q, const TensorD& t, int rows, int cols) {
  const unsigned bytes = (unsigned)((rows - 1) * (int)t.s1 + cols) * (unsigned)sizeof(T);
  return __builtin_amdgcn_make_buffer_rsrc((void*)const_cast<T*>(q), 0, bytes, 0x00027000);
}
// Lane's 16 values of column n of a (B,L,G|H,N)-shaped tensor, in the type they are stored in.
template <bool BF, typename T = typename std::conditional<BF, uint16_t, float>::type>
__device__ __forceinline__ void lane_load_raw(const TensorD& t, int b, int third, int n, bool vn, const RowMap& rm, T (&r)[16]) {
  const T* q = (const T*)t.ptr + ((long)b * t.s0 + (long)third * t.s2);
  // 32-bit offsets (the host checks that seqlen * stride fits): address = scalar base + per-lane offset.
  // ks is made opaque so that its multiples are formed here, next to their use, instead of being
  // hoisted out of an enclosing loop into (scarce) scalar registers.
  // BYTE offsets in 32 bits, so that the access is "scalar base + 32-bit per-lane offset" and costs one
  // integer add per element.
  const unsigned lo = (unsigned)(rm.base * (int)t.s1 + (rm.full || vn ? n : 0)) * (unsigned)sizeof(T);
  unsigned ks = (unsigned)(rm.step * (int)t.s1) * (unsigned)sizeof(T);
  ISSM_OPAQUE_S(ks);
  const char* qb = (const char*)q;
  if (rm.full) {
#pragma unroll
    for (int k = 0; k < 16; ++k) r[k] = *(const T*)(qb + (lo + (unsigned)(16 * (k >> 2) + (k & 3)) * ks));
  } else {
    const __amdgpu_buffer_rsrc_t rs = slab_of(q, t, rm.rows, rm.cols);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const unsigned o = lo + (unsigned)(16 * (k >> 2) + (k & 3)) * ks;
      if constexpr (BF) r[k] = __builtin_amdgcn_raw_buffer_load_b16(rs, o, 0, 0);
      else r[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0));
    }
  }
}
template <bool BF>
__device__ __forceinline__ void lane_load_ln(const TensorD& t, int b, int third, int n, bool vn, int g4,
                                             const RowMap& rm, float (&out)[16]) {
  typename std::conditional<BF, uint16_t, float>::type r[16];
  lane_load_raw<BF>(t, b, third, n, vn, rm, r);
#pragma unroll
  for (int k = 0; k < 16; ++k) out[k] = BF ? bf16_to_f((uint16_t)r[k]) : (float)r[k];
}
// Store of the lane's 16 values to column n of a (B,L,G|H,N)-shaped tensor (absent rows / columns skipped).
template <bool BF>
__device__ __forceinline__ void lane_store_ln(const TensorD& t, int b, int third, int n, bool vn, int g4,
                                              const RowMap& rm, const float (&v)[16]) {
  typedef typename std::conditional<BF, uint16_t, float>::type T;
  T* q = (T*)const_cast<void*>(t.ptr) + ((long)b * t.s0 + (long)third * t.s2);
  const unsigned lo = (unsigned)(rm.base * (int)t.s1 + n) * (unsigned)sizeof(T);
  unsigned ks = (unsigned)(rm.step * (int)t.s1) * (unsigned)sizeof(T);
  ISSM_OPAQUE_S(ks);
  char* qb = (char*)q;
  if (rm.full || !rm.edge) {  // uniform
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      T* d = (T*)(qb + (lo + (unsigned)(16 * (k >> 2) + (k & 3)) * ks));
      if (BF) *d = (T)f_to_bf16(v[k]); else *d = (T)v[k];
    }
  } else {
    const int rmax = vn ? rm.nvalid - 1 - 4 * g4 : -1;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int rk = 16 * (k >> 2) + (k & 3);
      if (rk <= rmax) {
        T* d = (T*)(qb + (lo + (unsigned)rk * ks));
        if (BF) *d = (T)f_to_bf16(v[k]); else *d = (T)v[k];
      }
    }
  }
}
// Lane's values of column n of a (P x N) fp32 slab: index q <-> row 16 (q >> 2) + 4 g4 + (q & 3).  `full`: every row
// exists; otherwise rows past the head dimension read its last row (they meet zero columns of the x / dy tiles).  Absent
// columns read column 0.
template <int CNT>
__device__ __forceinline__ void lane_load_pn(const float* __restrict__ src, int P, int N, int n, bool vn, int g4,
                                             bool full, float (&out)[CNT]) {
  const int nn = vn ? n : 0;
  const unsigned lo = (unsigned)(4 * g4 * N + nn) * 4u;
  unsigned nb = (unsigned)N * 4u;
  ISSM_OPAQUE_S(nb);
  const char* sb = (const char*)src;
  if (full) {
#pragma unroll
    for (int q = 0; q < CNT; ++q) out[q] = *(const float*)(sb + (lo + (unsigned)(16 * (q >> 2) + (q & 3)) * nb));
  } else {
    const unsigned last = (unsigned)((P - 1) * N + nn) * 4u;
#pragma unroll
    for (int q = 0; q < CNT; ++q) out[q] = *(const float*)(sb + min(lo + (unsigned)(16 * (q >> 2) + (q & 3)) * nb, last));
  }
}
// The lane's share of sum_p a[p] b[p] of two arrays as lane_load_pn leaves them (`full`: no row past the head dimension).
template <int CNT>
__device__ __forceinline__ float lane_dot_pn(const float (&a)[CNT], const float (&b)[CNT], int P, int g4, bool full) {
  float s = 0.0f;
#pragma unroll
  for (int q = 0; q < CNT; ++q) s += full || 16 * (q >> 2) + 4 * g4 + (q & 3) < P ? a[q] * b[q] : 0.0f;
  return s;
}
// dt transform (bias -> softplus -> clamp) of the lane's rows and the inclusive running sum of
// dt' * A * log2(e) down the chunk (so decays are exp2 of differences).  `raw` holds the loaded
// dt values.  dfac (if WANT_DFAC) receives d dt' / d dt: the softplus derivative times the clamp
// mask.  Returns the chunk total (running sum at row 63), the same on all lanes of the column.
// Per-column coefficients of the dt transform; loaded together with the column's dt values so that
// their latency is covered by the same prefetch.
struct Coef {
  float A, bias;
};
__device__ __forceinline__ Coef lane_coef(const KP& p, int h, int n, bool vn) {
  const int o = h * p.N + (vn ? n : 0);
  Coef c;
  c.A = p.A[o];
  c.bias = p.dt_bias ? p.dt_bias[o] : 0.0f;
  return c;
}
// dt transform of CNT values that already include the bias: softplus -> clamp; dfac (if WANT_DFAC) receives
// d dt' / d dt.  Softplus and its derivative share one exponential: with t = e^pre, softplus = log(1 + t) and
// sigmoid = t / (1 + t); above the reference's threshold of 20 both are replaced (identity, 1).  F_NOCLAMP: the limits
// are (0, inf) and softplus is on, so the clamp and its mask cannot act and are skipped.
template <bool WANT_DFAC, int CNT>
__device__ __forceinline__ void dt_transform(const KP& p, const float (&pre_)[CNT], float (&dtp)[CNT], float (&dfac)[CNT]) {
  if (p.flags & F_SOFTPLUS) {
    if (p.flags & F_NOCLAMP) {
#pragma unroll
      for (int k = 0; k < CNT; ++k) {
        const float pre = pre_[k];
        const float t = ex2(pre * LOG2E), u = 1.0f + t;
        const bool big = pre > 20.0f;
        dtp[k] = big ? pre : LN2 * __builtin_amdgcn_logf(u);
        if (WANT_DFAC) dfac[k] = big ? 1.0f : t * __builtin_amdgcn_rcpf(u);
      }
    } else {
#pragma unroll
      for (int k = 0; k < CNT; ++k) {
        const float pre = pre_[k];
        const float t = ex2(pre * LOG2E), u = 1.0f + t;
        const bool big = pre > 20.0f;
        const float sp = big ? pre : LN2 * __builtin_amdgcn_logf(u);
        dtp[k] = __builtin_amdgcn_fmed3f(sp, p.dt_min, p.dt_max);
        if (WANT_DFAC) dfac[k] = (sp < p.dt_min || sp > p.dt_max) ? 0.0f : (big ? 1.0f : t * __builtin_amdgcn_rcpf(u));
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < CNT; ++k) {
      const float sp = pre_[k];
      dtp[k] = __builtin_amdgcn_fmed3f(sp, p.dt_min, p.dt_max);
      if (WANT_DFAC) dfac[k] = (sp < p.dt_min || sp > p.dt_max) ? 0.0f : 1.0f;
    }
  }
}
// dt transform (bias -> softplus -> clamp) of the lane's 16 rows.  Rows past the end of the sequence and absent columns
// come out as dt' = 0 with derivative 0.
template <bool WANT_DFAC>
__device__ __forceinline__ void lane_dt(const KP& p, const Coef& cf, bool vn, int g4, const RowMap& rm,
                                        const float (&raw)[16], float (&dtp)[16], float (&dfac)[16]) {
  float pre[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) pre[k] = raw[k] + cf.bias;
  dt_transform<WANT_DFAC, 16>(p, pre, dtp, dfac);
  if (!rm.full && rm.edge) {  // uniform: rows past the end of the sequence and absent columns behave as dt' = 0
    const int lim = vn ? rm.nvalid - 4 * g4 : 0;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (16 * (k >> 2) + (k & 3) >= lim) {
        dtp[k] = 0.0f;
        if (WANT_DFAC) dfac[k] = 0.0f;
      }
  }
}
template <bool WANT_DFAC>
__device__ __forceinline__ float lane_prep(const KP& p, const Coef& cf, bool vn, int cm, int g4, const RowMap& rm,
                                           const float (&raw)[16], float (&dtp)[16], float (&cs)[16],
                                           float (&dfac)[16]) {
  const float A2 = cf.A * LOG2E;
  lane_dt<WANT_DFAC>(p, cf, vn, g4, rm, raw, dtp, dfac);
  // Running sum down the 64 rows: in the lane over its four rows of each tile, then across the four lane groups
  // of a tile, then across the tiles.  The cross-lane steps of the four tiles do not depend on each other, so each
  // step is issued for all four before any result is used (a cross-lane fetch goes through the LDS pipe: taken tile
  // by tile, twelve latencies would line up instead of three).  Same operations in the same order as tile by tile.
  float c[4], v[4], t[4];
  if (rm.full || rm.cut == 0) {  // uniform (and the only form the complete-tile variants contain)
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      float a = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a += dtp[4 * J + j] * A2;
        cs[4 * J + j] = a;
      }
      c[J] = a;
    }
  } else {  // packed sequences: the sum drops by SEQ_CUT at every row where the sequence id changes
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      const unsigned bits = (unsigned)(rm.cut >> (16 * J + 4 * g4)) & 15u;
      float a = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a += dtp[4 * J + j] * A2 - (((bits >> j) & 1u) ? SEQ_CUT : 0.0f);
        cs[4 * J + j] = a;
      }
      c[J] = a;
    }
  }
#pragma unroll
  for (int J = 0; J < 4; ++J) t[J] = __shfl_up(c[J], 16, 64);
#pragma unroll
  for (int J = 0; J < 4; ++J) v[J] = g4 >= 1 ? c[J] + t[J] : c[J];
#pragma unroll
  for (int J = 0; J < 4; ++J) t[J] = __shfl_up(v[J], 32, 64);
#pragma unroll
  for (int J = 0; J < 4; ++J) v[J] = g4 >= 2 ? v[J] + t[J] : v[J];  // inclusive over the lane groups
#pragma unroll
  for (int J = 0; J < 4; ++J) t[J] = __shfl(v[J], cm + 48, 64);      // tile totals
  float carry = 0.0f;
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    const float add = carry + (v[J] - c[J]);
#pragma unroll
    for (int j = 0; j < 4; ++j) cs[4 * J + j] += add;
    carry += t[J];
  }
  return carry;
}

// Running sums of a = dt' A log2(e) from the middle of the row's 32-row half of the chunk: pc[k] = sum of a over the rows of the
// half up to and including k's row, less half of the half's sum; half0, half1 = half of the halves' sums, tt[J] = a 16-row tile's
// (these the same on the four lanes of a column).  Used by the kernel that writes a decay exp2(cs[l] - cs[s]) as
// exp2(pc[l]) . exp2(-pc[s]) for rows of one half and with exp2(half0 + half1) between the two for rows of both: two exponentials
// per element and two per column serve every pair of rows of the chunk.
// LDS: the cross-lane steps through LDS (see group_sums).  (No packed sequences: that kernel does not take them.)
template <bool LDS>
__device__ __forceinline__ void lane_half_sums(float A2, int cm, int g4, const float (&dtp)[16], float (&pc)[16], float (&tt)[4],
                                               float& half0, float& half1) {
  float c[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    float a = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a += dtp[4 * J + j] * A2;
      pc[4 * J + j] = a;
    }
    c[J] = a;
  }
  float add[4];
  if constexpr (LDS) {
    float v[4], t[4];
#pragma unroll
    for (int J = 0; J < 4; ++J) t[J] = __shfl_up(c[J], 16, 64);
#pragma unroll
    for (int J = 0; J < 4; ++J) v[J] = g4 >= 1 ? c[J] + t[J] : c[J];
#pragma unroll
    for (int J = 0; J < 4; ++J) t[J] = __shfl_up(v[J], 32, 64);
#pragma unroll
    for (int J = 0; J < 4; ++J) v[J] = g4 >= 2 ? v[J] + t[J] : v[J];  // inclusive over the lane groups
#pragma unroll
    for (int J = 0; J < 4; ++J) tt[J] = __shfl(v[J], cm + 48, 64);    // tile totals
#pragma unroll
    for (int J = 0; J < 4; ++J) add[J] = v[J] - c[J];
  } else {
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      float after;
      group_sums(c[J], g4, add[J], after, tt[J]);
    }
  }
  half0 = 0.5f * (tt[0] + tt[1]);
  half1 = 0.5f * (tt[2] + tt[3]);
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    add[J] += ((J & 1) ? tt[J & 2] : 0.0f) - ((J & 2) ? half1 : half0);
#pragma unroll
    for (int j = 0; j < 4; ++j) pc[4 * J + j] += add[J];
  }
}

// v_mfma_f32_16x16x16_bf16: lane (m, g4) supplies k = 4 g4 .. 4 g4 + 3 -- in the column-lane layout exactly the lane's
// four rows of one 16-row tile.
typedef short sh4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f4 mfma_bf16k(bf4 a, bf4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(sh4, a), __builtin_bit_cast(sh4, b), c, 0, 0, 0);
}

// ------------------------------------------------------------------ cooperative tile loaders
// The unit's (64 x P) tile of a (B,L,H,P) tensor, zero padded to 16*PT columns: registers, then
// LDS dst[l][p] (leading dimension ld).  Element e = tid + 256 i is (l, p) = (e / 16PT, e % 16PT).
// Thread `tid` owns PT groups of four adjacent columns: group i is element e4 = tid + 256 i, i.e.
// (l, p) = (e4 / 4PT, 4 (e4 % 4PT)).  When the tensor allows it (uniform test) a group is one 8- or 16-byte
// access.
__device__ __forceinline__ bool lp_vec_ok(const KP& p, const TensorD& t, int esize) {
  return ((p.P & 3) == 0) && (((t.s0 | t.s1 | t.s2) & 3) == 0) && ((((uintptr_t)t.ptr) & (4 * esize - 1)) == 0);
}
template <bool BF, int PT, bool FULL = false>
__device__ __forceinline__ void lp_load(const KP& p, const Unit& u, const TensorD& t,
                                        float (&v)[CS * PT * 16 / NTHREADS], int tid = threadIdx.x) {
  constexpr int G4 = 4 * PT;  // groups per row
  typedef typename std::conditional<BF, uint16_t, float>::type T;
  const T* q = (const T*)t.ptr + ((long)u.b * t.s0 + (long)u.h * t.s2);
  const int nvalid = min(CS, p.L - u.c * CS);
  const long ss = (long)(u.dir ? -1 : 1) * t.s1;
  const long r0 = (long)(u.dir ? p.L - 1 - u.c * CS : u.c * CS) * t.s1;
  if (lp_vec_ok(p, t, sizeof(T))) {
    typedef typename std::conditional<BF, uint2, f4>::type V;
    V r[PT];
    bool ok[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
      ok[i] = p4 < p.P && (FULL || l < nvalid);
      r[i] = *(const V*)(q + (ok[i] ? r0 + l * ss + p4 : 0));
    }
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      if (BF) {
        const uint2 w = *(const uint2*)&r[i];
        v[4 * i + 0] = ok[i] ? __uint_as_float(w.x << 16) : 0.0f;
        v[4 * i + 1] = ok[i] ? __uint_as_float(w.x & 0xffff0000u) : 0.0f;
        v[4 * i + 2] = ok[i] ? __uint_as_float(w.y << 16) : 0.0f;
        v[4 * i + 3] = ok[i] ? __uint_as_float(w.y & 0xffff0000u) : 0.0f;
      } else {
        const f4 w = *(const f4*)&r[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * i + j] = ok[i] ? w[j] : 0.0f;
      }
    }
  } else {
    T r[4 * PT];
    bool ok[4 * PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ok[4 * i + j] = p4 + j < p.P && (FULL || l < nvalid);
        r[4 * i + j] = q[ok[4 * i + j] ? r0 + l * ss + p4 + j : 0];
      }
    }
#pragma unroll
    for (int e = 0; e < 4 * PT; ++e) v[e] = ok[e] ? (BF ? bf16_to_f((uint16_t)r[e]) : (float)r[e]) : 0.0f;
  }
}
// The tile in LDS as fp32, for reads of a column over four adjacent rows that differ from lane group to lane group: the groups'
// rows lie 16 banks apart, by four columns of padding or, four head tiles, by exchanging the row's 16-column pieces -- the 1 KB of
// padding would leave the kernels with (hi, lo) operand tiles beside it two workgroups a CU instead of three (16 x 2048 tokens, 16
// heads x 64, 512 states, both directions, fp32: k_chunk_scan 1030 -> 936 us, k_bwd_dx 1068 -> 960).
template <int PT>
struct RowTile {
  static constexpr int LD = PT == 4 ? 64 : PT * 16 + 4, SIZE = CS * LD;
  static __device__ __forceinline__ int at(int l, int p) { return l * LD + (PT == 4 ? p ^ ((l & 12) << 2) : p); }
};
template <int PT>
__device__ __forceinline__ void lp_store(const float (&v)[CS * PT * 16 / NTHREADS], float* dst, int tid = threadIdx.x) {
  constexpr int G4 = 4 * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e4 = tid + i * NTHREADS;
    *(f4*)(dst + RowTile<PT>::at(e4 / G4, (e4 % G4) * 4)) = (f4){v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
  }
}
// dy tile: from the caller's dout (io dtype) or from the gated fp32 (Bt,L,H,P) workspace copy.
template <bool BF, int PT, bool FULL = false>
__device__ __forceinline__ void dy_load(const KP& p, const Unit& u, const float* dy_ws,
                                        float (&v)[CS * PT * 16 / NTHREADS], int tid = threadIdx.x) {
  if (dy_ws) {
    TensorD t;
    t.ptr = dy_ws + (long)(u.bt - u.b) * p.L * p.H * p.P;  // so that b * s0 lands on row block bt
    t.s0 = (long)p.L * p.H * p.P;
    t.s1 = (long)p.H * p.P;
    t.s2 = p.P;
    lp_load<false, PT, FULL>(p, u, t, v, tid);
  } else {
    lp_load<BF, PT, FULL>(p, u, p.dout[u.dir], v, tid);
  }
}

// The same tiles for bf16 tensors as raw pairs of bf16 (no trip through fp32): group i of thread `tid` (lp_load's
// layout) in r[i], zeros where the row or the columns do not exist.  dy from the gated fp32 workspace is rounded here.
template <int PT, bool FULL>
__device__ __forceinline__ void lp_load_bf(const KP& p, const Unit& u, const TensorD& t, uint2 (&r)[PT], int tid) {
  if (lp_vec_ok(p, t, 2)) {
    constexpr int G4 = 4 * PT;
    const uint16_t* q = (const uint16_t*)t.ptr + ((long)u.b * t.s0 + (long)u.h * t.s2);
    const int nvalid = min(CS, p.L - u.c * CS);
    const long ss = (long)(u.dir ? -1 : 1) * t.s1;
    const long r0 = (long)(u.dir ? p.L - 1 - u.c * CS : u.c * CS) * t.s1;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
      const bool ok = p4 < p.P && (FULL || l < nvalid);
      const uint2 w = *(const uint2*)(q + (ok ? r0 + l * ss + p4 : 0));
      r[i] = ok ? w : make_uint2(0u, 0u);
    }
  } else {
    float v[CS * PT * 16 / NTHREADS];
    lp_load<true, PT, FULL>(p, u, t, v, tid);
#pragma unroll
    for (int i = 0; i < PT; ++i)  // exact: the values are bf16
      r[i] = make_uint2(pack_bf16(v[4 * i], v[4 * i + 1]), pack_bf16(v[4 * i + 2], v[4 * i + 3]));
  }
}
template <int PT, bool FULL>
__device__ __forceinline__ void dy_load_bf(const KP& p, const Unit& u, const float* dy_ws, uint2 (&r)[PT], int tid) {
  if (dy_ws) {
    float v[CS * PT * 16 / NTHREADS];
    dy_load<true, PT, FULL>(p, u, dy_ws, v, tid);
#pragma unroll
    for (int i = 0; i < PT; ++i)
      r[i] = make_uint2(pack_bf16(v[4 * i], v[4 * i + 1]), pack_bf16(v[4 * i + 2], v[4 * i + 3]));
  } else {
    lp_load_bf<PT, FULL>(p, u, p.dout[u.dir], r, tid);
  }
}
template <int PT, int LD>
__device__ __forceinline__ void lp_store_raw(const uint2 (&r)[PT], uint16_t* dst, int tid) {
  constexpr int G4 = 4 * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e4 = tid + i * NTHREADS;
    *(uint2*)(dst + (e4 / G4) * LD + (e4 % G4) * 4) = r[i];
  }
}

// Lower triangle (s <= l, rest zero) of a 64x64 fp32 block: registers, then LDS dst[l][s] (ld = LDC).
__device__ __forceinline__ void tril_load(const float* __restrict__ src, f4 (&v)[4], int tid = threadIdx.x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = tid + i * NTHREADS, l = e >> 4, s4 = (e & 15) * 4;
    v[i] = (s4 <= l) ? *(const f4*)(src + l * CS + s4) : (f4){0, 0, 0, 0};
  }
}
// The same lower triangle from the pair of symmetric bf16 matrices (hi at src, lo 8 KB behind it, each 64 x 64) that
// k_bwd_dstates writes for fp32 inputs: dM = hi + lo.
__device__ __forceinline__ void tril_load_hl(const float* __restrict__ src, f4 (&v)[4], int tid = threadIdx.x) {
  const uint16_t* hi = reinterpret_cast<const uint16_t*>(src);
  const uint16_t* lo = hi + CS * CS;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = tid + i * NTHREADS, l = e >> 4, s4 = (e & 15) * 4;
    const uint2 a = *(const uint2*)(hi + l * CS + s4), b = *(const uint2*)(lo + l * CS + s4);
    const f4 w = {__uint_as_float(a.x << 16) + __uint_as_float(b.x << 16),
                  __uint_as_float(a.x & 0xffff0000u) + __uint_as_float(b.x & 0xffff0000u),
                  __uint_as_float(a.y << 16) + __uint_as_float(b.y << 16),
                  __uint_as_float(a.y & 0xffff0000u) + __uint_as_float(b.y & 0xffff0000u)};
    v[i] = (s4 <= l) ? w : (f4){0, 0, 0, 0};
  }
}
__device__ __forceinline__ void tril_store(const f4 (&v)[4], float* dst, int tid = threadIdx.x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = tid + i * NTHREADS, l = e >> 4, s4 = (e & 15) * 4;
    f4 w = v[i];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s4 + j > l) w[j] = 0.0f;
    *(f4*)(dst + l * LDC + s4) = w;
  }
}

// Four adjacent fp32 values at any element offset (a type that only promises element alignment: unaligned accesses are
// legal on this target, and rows of N floats start anywhere when N is not a multiple of 4).
struct __attribute__((packed, aligned(4))) F4Any {
  float x, y, z, w;
};
__device__ __forceinline__ f4 ld_f4_any(const float* q) {
  const F4Any w = *(const F4Any*)q;
  return (f4){w.x, w.y, w.z, w.w};
}
__device__ __forceinline__ void st_f4_any(float* q, f4 v) {
  F4Any w;
  w.x = v[0]; w.y = v[1]; w.z = v[2]; w.w = v[3];
  *(F4Any*)q = w;
}

// Columns n0..n0+63 of a (P x N) fp32 slab: registers, then LDS dst[p][col] (leading dimension LDN).  Rows past P repeat
// the last one (what they contribute to is not stored).  Columns past N read whatever follows in the slab, or zero beyond
// its end (a raw buffer load checks every dword; it needs dword alignment only): pn_edge, called before the values are used,
// zeroes them.
template <int PT>
struct PnRegs {
  static constexpr int Q = NS / 4, TOT = PT * 16 * Q, CNT = (TOT + NTHREADS - 1) / NTHREADS;
  static_assert(TOT % NTHREADS == 0, "every thread owns CNT quads");
  f4 v[CNT];
};
template <int PT, bool FULL>
__device__ __forceinline__ void pn_load(const KP& p, const float* __restrict__ src, int n0, PnRegs<PT>& r,
                                        int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
  const int c = n0 + (tid % R::Q) * 4;
  if constexpr (FULL) {
#pragma unroll
    for (int i = 0; i < R::CNT; ++i)
      r.v[i] = *(const f4*)(src + (min((tid + i * NTHREADS) / R::Q, p.P - 1) * p.N + c));
  } else {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)const_cast<float*>(src), 0, (unsigned)(p.P * p.N) * 4u, 0x00027000);
#pragma unroll
    for (int i = 0; i < R::CNT; ++i) {
      const u4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, (min((tid + i * NTHREADS) / R::Q, p.P - 1) * p.N + c) * 4, 0, 0);
      r.v[i] = __builtin_bit_cast(f4, w);
    }
  }
}
template <int PT>
__device__ __forceinline__ void pn_edge(const KP& p, int n0, PnRegs<PT>& r, int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
  if (n0 + NS <= p.N) return;  // uniform
  const int left = p.N - n0 - (tid % R::Q) * 4;   // columns of the quad that exist
#pragma unroll
  for (int i = 0; i < R::CNT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j >= left) r.v[i][j] = 0.0f;
}
template <int PT>
__device__ __forceinline__ void pn_store(const PnRegs<PT>& r, float* dst, int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
#pragma unroll
  for (int i = 0; i < R::CNT; ++i) {
    const int e = tid + i * NTHREADS, pp = e / R::Q, c4 = (e % R::Q) * 4;
    if (e < R::TOT) *(f4*)(dst + pp * LDN + c4) = r.v[i];
  }
}

// Index helpers for the fp32 intermediates.
//   states  (Bt, nc+1, H, P, N): slot c = state entering chunk c, slot nc = final state
//   dstates (Bt, nc,   H, P, N)
//   per-chunk vectors (Bt, nc, H, N); square blocks (Bt, nc, H, 64, 64)
__device__ __forceinline__ long st_off(const KP& p, int bt, int c, int h) {
  return (((long)bt * (p.nc + 1) + c) * p.H + h) * p.P * p.N;
}
__device__ __forceinline__ long dst_off(const KP& p, int bt, int c, int h) {
  return (((long)bt * p.nc + c) * p.H + h) * p.P * p.N;
}
__device__ __forceinline__ long vec_off(const KP& p, int bt, int c, int h) {
  return (((long)bt * p.nc + c) * p.H + h) * p.N;
}
__device__ __forceinline__ long sq_off(const KP& p, int bt, int c, int h) {
  return (((long)bt * p.nc + c) * p.H + h) * CS * CS;
}

// Kernel dispatch on (P tiles, io dtype, dt dtype, complete tiles or not): the statement sees PT_, IOB_, DTB_, FULL_ as
// constants.
#define ISSM_DISPATCH_FULL(full, ...)                              \
  if (full) { constexpr bool FULL_ = true; __VA_ARGS__ }           \
  else { constexpr bool FULL_ = false; __VA_ARGS__ }
#define ISSM_DISPATCH_DT(iob, dtb, full, ...)                          \
  if (iob) {                                                           \
    constexpr bool IOB_ = true;                                        \
    if (dtb) { constexpr bool DTB_ = true; ISSM_DISPATCH_FULL(full, __VA_ARGS__) }  \
    else { constexpr bool DTB_ = false; ISSM_DISPATCH_FULL(full, __VA_ARGS__) }     \
  } else {                                                             \
    constexpr bool IOB_ = false;                                       \
    if (dtb) { constexpr bool DTB_ = true; ISSM_DISPATCH_FULL(full, __VA_ARGS__) }  \
    else { constexpr bool DTB_ = false; ISSM_DISPATCH_FULL(full, __VA_ARGS__) }     \
  }
#define ISSM_DISPATCH(p, ...)                                                                        \
  do {                                                                                               \
    const int pt_ = ((p).P + 15) / 16;                                                               \
    const bool iob_ = (p).io_dt != 0, dtb_ = (p).dt_dt != 0;                                         \
    const int full_ = (p).full_tiles;                                                                \
    if (pt_ <= 2) { constexpr int PT_ = 2; ISSM_DISPATCH_DT(iob_, dtb_, full_, __VA_ARGS__) }        \
    else if (pt_ == 3) { constexpr int PT_ = 3; ISSM_DISPATCH_DT(iob_, dtb_, full_, __VA_ARGS__) }   \
    else { constexpr int PT_ = 4; ISSM_DISPATCH_DT(iob_, dtb_, full_, __VA_ARGS__) }                 \
  } while (0)

}  // namespace issm
