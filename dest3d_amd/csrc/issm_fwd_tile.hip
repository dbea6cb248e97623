// k_local_tile: the chunk-local pass of the forward (dt transform, running sums, chunk end states S_c, intra-chunk
// matrix M_c, the chunk's total decay) in a ROW-lane layout.
//
// Lane (i, kg) of a wave owns row i of every 16-row tile of the chunk and four adjacent state columns
// n = n0 + 4 kg .. + 3: exactly the operand layout of v_mfma_f32_16x16x16_bf16 for a contraction over the state
// columns, and 16 bytes (fp32) or 8 (bf16) per tensor and tile.  Four lanes that follow one another in a wave request one row's 16 columns, and
// the wave hands the pieces over to the lanes that work on them (row_pieces_to_lanes).  The four waves of a workgroup take the
// four 16-column quarters of each 64-column step.  A step's operands are requested when the step before has used its own, in
// one stretch of code without branches, so that a wait is for the request it needs and not for the stores behind it.
//   Requests by row pieces, those waits, and no copies of what was requested: 8 x 1024 tokens, both directions, 8 heads x 32, 256 states, fp32 91
// -> 82 us; heads of 36, bf16 84 -> 66; 2 x 16384, one direction, bf16 188 -> 150; 16 x 2048, both, 16 heads x 64, 512 states, fp32 1463 -> 1303.
//
//   running sums   down the 16 rows of a tile = across the 16 lanes of a DPP row: four shifted adds per value.
//                  pc[l] = sum of a = dt' A log2(e) over the rows of l's tile up to and including l.
//   decays         exp2(cs[l] - cs[s]) = up[l] . G . iup[s],  up = exp2(pc), iup = exp2(-pc), G = product of the whole-
//                  tile decays et[K] = exp2(tile sum K) of the tiles from s's tile up to (not including) l's tile
//   M (I, J)       = sum_n U_I[l][n] X_IJ[s][n],  U = C up,  X_JJ = W = dt' B iup,  X_(J+1)J = V = W et[J],
//                  X_(J+2)J = V et[J+1],  X_30 = V et[1] et[2]: ten plain 16 x 16 products per 16 columns with both
//                  operands taken from registers as they are.  Each wave sums over its columns; the four partial sums
//                  meet in LDS once per chunk.
//   S^T (n, p)     = sum_l V[l][n] (decay from the end of l's tile to the end of the chunk)[n] x[l][p].  This contracts
//                  over the ROWS, so V is needed with the roles of lane and register exchanged: one matrix instruction
//                  against a 16 x 16 identity moves a (bf16, hence exactly representable) tile into the accumulator
//                  layout, which is that exchanged layout.  x^T comes from LDS.  The decay to the end of the chunk depends
//                  on the OUTPUT row n only: the accumulator is multiplied by et[J+1] between the tiles (Horner).  The
//                  result holds four adjacent columns of a state row per lane: 16-byte stores.
//
// Everything but W is a product of factors <= 1.  W grows like 2^(span of a tile) and is taken where every tile of the wave's
// columns decays by less than 2^FWD_SPAN_LIMIT.
//   A chunk with another tile is computed once more, by the same workgroup, with the level-hierarchy body (k_chunk_local_body),
//   which has no such limit and overwrites everything written for the chunk before.  bf16 inputs: the wave that meets such a
//   tile raises a flag that all look at once a step, and the rest of the steps is left out (a quarter of the chunks of a freshly
//   initialised decoder, 8 x 1024 tokens, 256 queries: 195 -> 179 us a layer, 118 without a device-wide fence).  fp32 inputs, whose operand pairs leave no
//   registers to spare, pay for the look: 1505 -> 1575 us at 16 x 2048 tokens, 16 heads x 64, 512 states, nothing out of range.
//   ANY, bf16 inputs of calls that nothing is differentiated through: the first step with such a tile is left by the loop over the steps,
// and it and all that follow are evaluated, by its wave alone, in a loop of their own, with the diagonal blocks in parts whose factors are all
// <= 1 (far_diagonal) and V from its own exponential.  A freshly initialised decoder has such tiles in 16 % of its chunks and heads, there
// mostly in all steps, and those workgroups decide when the launch ends: 1024 tokens, 256 queries 20.9 us a layer (36 with the chunk computed once
// more; 22.1 with the loop over the steps left at a step's end, its operands masked so that it adds nothing).  As
// accurate as the level form, but rounded elsewhere, and through six layers the gradients move by up to 0.8 of their mean square between the
// two: training keeps the level form (8 x 1024 tokens: 155 us, 110 with this one).
#include "issm_dev.h"
#include "issm_fwd_local.h"

namespace issm {

constexpr float FWD_SPAN_LIMIT = 100.0f;

template <int PT, bool SPLIT>
struct FwdTileSmem {
  static constexpr int LDT = CS + 8;   // row stride of the transposed x tile
  uint16_t xt_hi[PT * 16 * LDT];       // x tile transposed, [p][l]
  uint16_t xt_lo[SPLIT ? PT * 16 * LDT : 8];
  f4 red[4 * 10 * 64];                 // the four waves' partial sums of the ten blocks of M; before, each wave's part serves row_pieces_to_lanes
  int bad;                             // not ANY: some tile is out of range
};
template <int PT, bool SPLIT, bool ANY>
constexpr size_t fwd_tile_lds() {     // not ANY: the level-hierarchy body lays its own structure over the same memory
  return !ANY && sizeof(FwdTileSmem<PT, SPLIT>) < sizeof(FwdLocalSmem<PT, SPLIT>) ? sizeof(FwdLocalSmem<PT, SPLIT>)
                                                                                   : sizeof(FwdTileSmem<PT, SPLIT>);
}

// inclusive running sums over the 16 lanes of a DPP row (lanes sharing lane >> 4) of 16 values, step by step for all of them: an instruction
// that reads another lane's value waits for two others behind the one that wrote it
template <int CTRL>
__device__ __forceinline__ void row_add(float (&v)[16]) {   // lanes without a source add 0
#pragma unroll
  for (int k = 0; k < 16; ++k)
    v[k] += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v[k]), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ void row_scans(float (&v)[16]) {
  row_add<0x111>(v);  // row_shr:1
  row_add<0x112>(v);
  row_add<0x114>(v);
  row_add<0x118>(v);
}

// the value of lane J of a DPP row, on its 16 lanes
template <int J>
__device__ __forceinline__ float row_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + J, 0xf, 0xf, true));
}

// one of each four lanes' values (a DPP quad permutation)
template <int PERM>
__device__ __forceinline__ float quad_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), PERM, 0xf, 0xf, true));
}

// four fp32 accumulator values that are exact bf16 numbers -> a bf16 fragment
__device__ __forceinline__ bf4 exact_bf4(f4 v) {
  // v_perm_b32: bytes 2, 3 of the second source below bytes 2, 3 of the first
  const uint2 r = make_uint2(__builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u),
                             __builtin_amdgcn_perm(__float_as_uint(v[3]), __float_as_uint(v[2]), 0x07060302u));
  return __builtin_bit_cast(bf4, r);
}

template <bool SPLIT>
struct Frag {
  bf4 h, l;
};
template <bool SPLIT>
__device__ __forceinline__ Frag<SPLIT> make_frag(float a, float b, float c, float d) {
  Frag<SPLIT> f;
  const float v[4] = {a, b, c, d};
  if (SPLIT) {
    split4(v, f.h, f.l);
  } else {
    const uint2 r = make_uint2(pack_bf16(a, b), pack_bf16(c, d));
    f.h = __builtin_bit_cast(bf4, r);
    f.l = f.h;
  }
  return f;
}
// acc += A . B^T over the lane groups' columns: both operands (hi, lo) pairs when SPLIT, one bf16 rounding otherwise
template <bool SPLIT>
__device__ __forceinline__ f4 frag_product(const Frag<SPLIT>& a, const Frag<SPLIT>& b, f4 acc) {
  if (SPLIT) {
    acc = mfma_bf16k(a.l, b.h, acc);
    acc = mfma_bf16k(a.h, b.l, acc);
  }
  return mfma_bf16k(a.h, b.h, acc);
}

// Four adjacent elements at any element offset (one wide access: unaligned ones are legal on this target).
struct __attribute__((packed, aligned(2))) Bf4Any {
  unsigned x, y;
};
template <bool BF>
struct RawVec {
  typedef typename std::conditional<BF, Bf4Any, F4Any>::type type;
};
template <bool BF>
__device__ __forceinline__ void unpack4(const typename RawVec<BF>::type& r, float* out) {
  if constexpr (BF) {
    out[0] = __uint_as_float(r.x << 16);
    out[1] = __uint_as_float(r.x & 0xffff0000u);
    out[2] = __uint_as_float(r.y << 16);
    out[3] = __uint_as_float(r.y & 0xffff0000u);
  } else {
    out[0] = r.x; out[1] = r.y; out[2] = r.z; out[3] = r.w;
  }
}

// What the lanes of a wave have requested -- lane 4 r + q the columns 4 q .. + 3 of row r, so that four neighbours' accesses are one
// piece of memory -- to those that work on it, through LDS that no other wave uses.  Piece 4 r + q lies in slot 4 r + (q ^ turn): those of one q,
// read together, are in different banks.  (Requested by the lanes that work on it, an instruction's 64 lanes were 64 look-ups in the L1
// instead of 16: 148 thousand of them a CU, which the kernel waited for in its 165 thousand cycles, at the first size above, vector issue 59 % of
// the cycles; 57 thousand now, and vector issue 71 %.  By itself the change gave 91 -> 83 us fp32 and 84 -> 70 bf16, heads of 36.)
template <typename Raw>
__device__ __forceinline__ void row_pieces_to_lanes(const Raw (&raw)[4], void* area, int lane, float (&v)[16]) {
  constexpr bool BF = sizeof(Raw) == 8;
  typedef typename std::conditional<BF, uint2, f4>::type Plain;
  typedef Plain __attribute__((may_alias)) Slot;
  Slot* q = (Slot*)area;
  auto slot = [](int r, int c) { return 4 * r + (c ^ (BF ? (r >> 3) * 2 : r >> 2)); };
  const int from = slot(lane >> 2, lane & 3), to = slot(lane & 15, lane >> 4);
#pragma unroll
  for (int J = 0; J < 4; ++J) q[64 * J + from] = __builtin_bit_cast(Plain, raw[J]);
#pragma unroll
  for (int J = 0; J < 4; ++J) unpack4<BF>(__builtin_bit_cast(Raw, (Plain)q[64 * J + to]), v + 4 * J);
}

// FULLP: the head dimension fills its tiles.  EDGE: chunks with fewer than 64 rows and steps with fewer than 64 columns
// may exist (N >= 4).  A lane's rows past the end read the chunk's last one and get dt' = 0, as do whole lanes past the last
// column; a lane whose four columns cross it works on columns N - 4 .. N - 1 instead, those its neighbour owns with dt' = 0
// and not stored.  The diagonal blocks of M take fp32 matrix instructions: the level form, which evaluates such calls
// wherever this kernel cannot, has the pairs inside groups of four rows in fp32, and what a pair is computed in is not to
// depend on the kernel.  (Those entries of M: 2.4e-3 from float64 with operands rounded once to bf16, 4.4e-6 as bf16 pairs,
// 2.6e-7 like this.  8 x 1024 tokens, 8 heads x 32, N = 250: fp32 55.4 us with pairs, 55.8 like this; bf16 43.4 and 46.9.)
// ANY (bf16 inputs): tiles of any decay within the loop's own pass.
template <int PT, bool IOB, bool DTB, bool FULLP, bool EDGE, bool ANY>
__global__ __launch_bounds__(NTHREADS, 2) void k_local_tile(KP p, float* __restrict__ states, float* __restrict__ cs_last,
                                                            float* __restrict__ cabt) {
  warm_args();
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr bool SPLIT = !IOB;
  typedef FwdTileSmem<PT, SPLIT> SM;
  SM& s = *reinterpret_cast<SM*>(smem_raw);
  constexpr int LDT = SM::LDT;
  typedef typename RawVec<DTB>::type RawDt;
  typedef typename RawVec<IOB>::type RawIo;
  typedef typename std::conditional<DTB, uint16_t, float>::type TDt;
  typedef typename std::conditional<IOB, uint16_t, float>::type TIo;
  typedef Frag<SPLIT> Fr;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kg = lane >> 4;
  const int ri = lane >> 2, rkg = lane & 3;   // the row and the columns that the lane requests
  const int uidx = xcd_remap(blockIdx.x, gridDim.x);
  const Unit u = decode_unit(p, uidx);

  // addresses: uniform base + per-lane 32-bit element offset (the host checks that seqlen * stride fits in 31 bits);
  // tile J lies 16 J rows further along the scan, the step's columns 64 further along the row
  const int tl = u.dir ? p.L - 1 - u.c * CS - ri : u.c * CS + ri;   // the token of tile 0 whose operands the lane requests
  const int sgn = u.dir ? -1 : 1;
  const int nvalid = EDGE ? min(CS, p.L - u.c * CS) : CS;
  const int ncol = 16 * w + 4 * kg, rcol = 16 * w + 4 * rkg;       // the lane's first column within a step, and of what it requests
  const TDt* qdt = (const TDt*)p.dt.ptr + ((long)u.b * p.dt.s0 + (long)u.h * p.dt.s2);
  const TIo* qB = (const TIo*)p.Bm[u.dir].ptr + ((long)u.b * p.Bm[u.dir].s0 + (long)u.g * p.Bm[u.dir].s2);
  const TIo* qC = (const TIo*)p.Cm[u.dir].ptr + ((long)u.b * p.Cm[u.dir].s0 + (long)u.g * p.Cm[u.dir].s2);
  // element offsets of the lane's rows.  Complete tiles: tile J lies a uniform distance behind tile 0, so one register per
  // tensor; otherwise a row past the end is the chunk's last one, and each tile has its own.
  const int sdt = (int)p.dt.s1, sB = (int)p.Bm[u.dir].s1, sC = (int)p.Cm[u.dir].s1;
  constexpr int NO = EDGE ? 4 : 1;
  unsigned odt[NO], oB[NO], oC[NO];
#pragma unroll
  for (int J = 0; J < NO; ++J) {
    const int t = EDGE ? tl + sgn * (min(16 * J + ri, nvalid - 1) - ri) : tl;
    odt[J] = (unsigned)(t * sdt + (EDGE ? 0 : rcol));
    oB[J] = (unsigned)(t * sB + (EDGE ? 0 : rcol));
    oC[J] = (unsigned)(t * sC + (EDGE ? 0 : rcol));
  }
  const int jdt = EDGE ? 0 : sgn * 16 * sdt, jB = EDGE ? 0 : sgn * 16 * sB, jC = EDGE ? 0 : sgn * 16 * sC;
  const float* qA = p.A + u.h * p.N;
  const float* qbias = (p.dt_bias ? p.dt_bias : p.A) + u.h * p.N;  // without a bias: any valid address, scaled by 0
  const float bias_on = p.dt_bias ? 1.0f : 0.0f;

  RawDt rdt[4];
  RawIo rB[4], rC[4];
  F4Any rA, rbias;
#define ISSM_REQUEST_DT(n0_)                                                           \
  {                                                                                    \
    const int c_ = EDGE ? min((n0_) + rcol, p.N - 4) : (n0_);                          \
    const int a_ = EDGE ? min((n0_) + ncol, p.N - 4) : (n0_) + ncol;                   \
    _Pragma("unroll") for (int J = 0; J < 4; ++J)                                      \
      rdt[J] = *(const RawDt*)(qdt + (int)(odt[J % NO] + (unsigned)(J * jdt + c_)));   \
    rA = *(const F4Any*)(qA + a_);                                                     \
    rbias = *(const F4Any*)(qbias + a_);                                               \
  }
#define ISSM_REQUEST_B(n0_)                                                            \
  {                                                                                    \
    const int c_ = EDGE ? min((n0_) + rcol, p.N - 4) : (n0_);                          \
    _Pragma("unroll") for (int J = 0; J < 4; ++J)                                      \
      rB[J] = *(const RawIo*)(qB + (int)(oB[J % NO] + (unsigned)(J * jB + c_)));       \
  }
#define ISSM_REQUEST_C(n0_)                                                            \
  {                                                                                    \
    const int c_ = EDGE ? min((n0_) + rcol, p.N - 4) : (n0_);                          \
    _Pragma("unroll") for (int J = 0; J < 4; ++J)                                      \
      rC[J] = *(const RawIo*)(qC + (int)(oC[J % NO] + (unsigned)(J * jC + c_)));       \
  }
#define ISSM_REQUEST(n0_)                                                              \
  {                                                                                    \
    ISSM_REQUEST_DT(n0_)                                                               \
    ISSM_REQUEST_C(n0_)                                                                \
    ISSM_REQUEST_B(n0_)                                                                \
  }
  ISSM_REQUEST(0);

  // the unit's x tile, transposed, as bf16 (hi, lo) in LDS (its loads travel together with the first step's above)
  {
    float xv[CS * PT * 16 / NTHREADS];
    lp_load<IOB, PT, !EDGE>(p, u, p.x[u.dir], xv);
    lp_store_split_t<PT, LDT, SPLIT>(xv, s.xt_hi, s.xt_lo);
  }


  auto hand_over = [&](const auto& raw, float (&v)[16]) __attribute__((always_inline)) { row_pieces_to_lanes(raw, s.red + w * 640, lane, v); };

  // identity operand of the exchange of lane and register roles: B[k = 4 kg + r][j = i] = (k == j)
  bf4 ident;
  {
    const unsigned one = 0x3F80u;
    const int r1 = i - 4 * kg;
    const uint2 idr = make_uint2((r1 == 0 ? one : 0u) | (r1 == 1 ? one << 16 : 0u), (r1 == 2 ? one : 0u) | (r1 == 3 ? one << 16 : 0u));
    ident = __builtin_bit_cast(bf4, idr);
  }

  // Diagonal block of a tile whose decays may be out of range: pairs of rows in different halves, then in different quarters
  // of a half, each with the row between the two as the reference -- both factors of every pair are <= 1 -- and in fp32 those
  // inside a quarter (four rows), with its second row as the reference or, where that is out of range too, in three parts.
  auto far_diagonal = [&](const float* c4, const float* w4, const float* pc4, f4& m) __attribute__((always_inline)) {
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float uu[4], ww[4];
    {
      const bool up8 = i & 8;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d = pc4[r] - row_lane<7>(pc4[r]), e = ex2(up8 ? d : -d);
        uu[r] = up8 ? c4[r] * e : 0.0f;
        ww[r] = up8 ? 0.0f : w4[r] * e;
      }
      m = frag_product<SPLIT>(make_frag<SPLIT>(uu[0], uu[1], uu[2], uu[3]), make_frag<SPLIT>(ww[0], ww[1], ww[2], ww[3]), m);
    }
    {
      const bool up4 = i & 4;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float lo = row_lane<3>(pc4[r]), hi = row_lane<11>(pc4[r]);
        const float d = pc4[r] - (i & 8 ? hi : lo), e = ex2(up4 ? d : -d);
        uu[r] = up4 ? c4[r] * e : 0.0f;
        ww[r] = up4 ? 0.0f : w4[r] * e;
      }
      const f4 t = frag_product<SPLIT>(make_frag<SPLIT>(uu[0], uu[1], uu[2], uu[3]), make_frag<SPLIT>(ww[0], ww[1], ww[2], ww[3]), zero);
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] += kg == 3 && i < 4 ? 0.0f : t[r];   // (rows of different halves: not from here)
    }
    float d[4], dmin = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      d[r] = pc4[r] - quad_lane<0x55>(pc4[r]);   // lane 1 of four
      dmin = fminf(dmin, -fabsf(d[r]));
    }
    if (__ballot(!(dmin >= -FWD_SPAN_LIMIT)) == 0ull) {
      f4 t = zero;
#pragma unroll
      for (int r = 0; r < 4; ++r) t = mfma4(c4[r] * ex2(d[r]), w4[r] * ex2(-d[r]), t);
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] += kg == i >> 2 ? t[r] : 0.0f;
    } else {
      f4 t = zero;   // rows 2, 3 with rows 0, 1
      const bool up2 = i & 2, up1 = i & 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = ex2(up2 ? d[r] : -d[r]);
        t = mfma4(up2 ? c4[r] * e : 0.0f, up2 ? 0.0f : w4[r] * e, t);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] += kg == i >> 2 ? t[r] : 0.0f;
      t = zero;      // 1 with 0, 3 with 2
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = ex2(quad_lane<0xf5>(pc4[r]) - pc4[r]);   // lanes 1, 1, 3, 3
        t = mfma4(up1 ? c4[r] : 0.0f, up1 ? 0.0f : w4[r] * e, t);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] += 4 * kg + r == i + 1 ? t[r] : 0.0f;
      t = zero;      // a row with itself
#pragma unroll
      for (int r = 0; r < 4; ++r) t = mfma4(c4[r], w4[r], t);
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] += 4 * kg + r == i ? t[r] : 0.0f;
    }
  };

  f4 macc[10];
#pragma unroll
  for (int q = 0; q < 10; ++q) macc[q] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
  float etmin = 1.0f;  // smallest whole-tile decay seen by the lane
  const float thr = ex2(-FWD_SPAN_LIMIT);

  if (tid == 0) s.bad = 0;
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0).  (What is under way here the waits in the loop would count with their own, as the compiler
                                        // merges the two: the one at its head then waited for everything, the stores of the step before among it.)
  __syncthreads();  // x tile complete
  float* sdst = states + st_off(p, u.bt, u.c, u.h);
  const __amdgpu_buffer_rsrc_t slab = __builtin_amdgcn_make_buffer_rsrc(sdst, 0, (unsigned)(p.P * p.N) * 4u, 0x00027000);
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  float* cdst = cs_last + vec_off(p, u.bt, u.c, u.h);

  // not ANY, a tile was out of range: the loop ends with the step.  (With a second way out of it, in the middle of a step, every wait at its
  // head counts on a step broken off there and waits for all that is under way, the step's own stores among it.)
  bool stop = false;
  if constexpr (!ANY) {
    constexpr bool DEEP = false;
#pragma unroll 1
    for (int n0 = 0; (n0 < p.N) & !stop; n0 += NS) {
#include "issm_fwd_tile_step.h"
    }
  } else {
    int n0 = 0;
#pragma unroll 1
    for (; n0 < p.N; n0 += NS) {
      constexpr bool DEEP = false;
#include "issm_fwd_tile_step.h"
    }
    if (n0 < p.N) {
      asm volatile("");   // keeps the two loops apart
      ISSM_REQUEST(n0);
#pragma unroll 1
      for (; n0 < p.N; n0 += NS) {
        constexpr bool DEEP = true;
#include "issm_fwd_tile_step.h"
      }
    }
  }
#undef ISSM_REQUEST
#undef ISSM_REQUEST_C
#undef ISSM_REQUEST_B
#undef ISSM_REQUEST_DT

  // ---- M: the waves' partial sums meet in LDS; wave w then finishes blocks w, w + 4, w + 8
#pragma unroll
  for (int q = 0; q < 10; ++q) s.red[(w * 10 + q) * 64 + lane] = macc[q];
  if (!IOB && __ballot(!(etmin >= thr)) != 0ull) s.bad = 1;
  __syncthreads();
  const int anybad = ANY ? 0 : s.bad;  // uniform
  float* m = cabt + sq_off(p, u.bt, u.c, u.h);
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const int q = w + 4 * t;  // uniform
    if (q < 10) {
      f4 v = s.red[q * 64 + lane];
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) {
        const f4 o = s.red[(ww * 10 + q) * 64 + lane];
        v[0] += o[0]; v[1] += o[1]; v[2] += o[2]; v[3] += o[3];
      }
      // block (I, J) of index q: 0..3 diagonal, 4..6 (J+1, J), 7..8 (J+2, J), 9 (3, 0)
      const int I = q < 4 ? q : q < 7 ? q - 3 : q < 9 ? q - 5 : 3, J = q < 4 ? q : q < 7 ? q - 4 : q < 9 ? q - 7 : 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int l = 4 * kg + r;  // accumulator r <-> (row 4 kg + r, column i) of the block
        m[(16 * I + l) * CS + 16 * J + i] = (I == J && i > l) ? 0.0f : v[r];
      }
    }
  }
  if (!ANY && anybad) {
    // A tile of this chunk decays by more than 2^-FWD_SPAN_LIMIT: everything is computed once more in the form that has no
    // such limit.  Its stores go to places that other waves of this workgroup have stored to above: those stores have reached the
    // L2, which all of the workgroup's waves share, before the barrier.  (A device-wide fence in its place writes back and
    // invalidates the XCD's L2 once a wave of every such chunk, under all the other workgroups: layers of 8 x 1024 tokens, 8 heads
    // x 36, 256 states, bf16 with 5, 12, 16, 35 and 48 % of their chunks out of range took 119, 146, 163, 205 and 236 us, and
    // take 104, 108, 119, 118 and 126.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (!ANY) k_chunk_local_body<PT, IOB, DTB, !EDGE>(p, states, cs_last, cabt);
  }
}

// Whether the row-lane kernel takes the launch: both outputs wanted, four columns to work on, no packed sequences (their
// cuts are outside the form's range).
bool local_tile_available(const KP& p, const float* states, const float* cabt) {
  return !p.seq_idx && p.N >= 4 && states && cabt;
}

template <typename K>
static int set_lds_tile(K kernel, size_t bytes) {   // (up to 64 KB needs no asking)
  return bytes > 64 * 1024 ? (int)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) : 0;
}

int launch_local_tile(const KP& p, float* states, float* cs_last, float* cabt, bool any, hipStream_t st) {
  const int units = p.B * p.ndir * p.nc * p.H;
  const int pt = (p.P + 15) / 16;
  // EDGE unless every tile is complete and every operand starts its rows at a multiple of four elements (16-byte stores of
  // the states and decay totals; operands elsewhere belong to the calls the level form's precision is kept for, see EDGE)
  auto rows_of_four = [](const TensorD& t, int bf) {
    return ((t.s0 | t.s1 | t.s2) & 3) == 0 && ((uintptr_t)t.ptr & (bf ? 7 : 15)) == 0;
  };
  bool edge = !p.full_tiles || !rows_of_four(p.dt, p.dt_dt) ||
              (((uintptr_t)states | (uintptr_t)cs_last | (uintptr_t)p.A | (uintptr_t)p.dt_bias) & 15);
  for (int d = 0; d < p.ndir; ++d) edge = edge || !rows_of_four(p.Bm[d], p.io_dt) || !rows_of_four(p.Cm[d], p.io_dt);
#define ISSM_LT_FORM(PT_, IOB_, DTB_, FULLP_, EDGE_, ANY_)                                                  \
  {                                                                                                         \
    constexpr auto kern = &k_local_tile<PT_, IOB_, DTB_, FULLP_, EDGE_, ANY_>;                              \
    constexpr size_t sm = fwd_tile_lds<PT_, !IOB_, ANY_>();                                                 \
    if (int e = set_lds_tile(kern, sm)) return e;                                                           \
    hipLaunchKernelGGL(kern, dim3(units), dim3(NTHREADS), sm, st, p, states, cs_last, cabt);                \
  }
#define ISSM_LT_ONE(PT_, IOB_, DTB_, FULLP_, EDGE_)                                                         \
  {                                                                                                         \
    if (IOB_ && any) ISSM_LT_FORM(PT_, IOB_, DTB_, FULLP_, EDGE_, IOB_)                                     \
    else ISSM_LT_FORM(PT_, IOB_, DTB_, FULLP_, EDGE_, false)                                                \
  }
#define ISSM_LT(PT_, IOB_, DTB_)                                                                            \
  {                                                                                                         \
    if (edge) ISSM_LT_ONE(PT_, IOB_, DTB_, false, true)                                                     \
    else if (p.P == 16 * PT_) ISSM_LT_ONE(PT_, IOB_, DTB_, true, false)                                     \
    else ISSM_LT_ONE(PT_, IOB_, DTB_, false, false)                                                         \
  }
#define ISSM_LT_DT(PT_)                                                      \
  {                                                                          \
    if (p.io_dt) {                                                           \
      if (p.dt_dt) ISSM_LT(PT_, true, true) else ISSM_LT(PT_, true, false)   \
    } else {                                                                 \
      if (p.dt_dt) ISSM_LT(PT_, false, true) else ISSM_LT(PT_, false, false) \
    }                                                                        \
  }
  if (pt <= 2) ISSM_LT_DT(2) else if (pt == 3) ISSM_LT_DT(3) else ISSM_LT_DT(4)
#undef ISSM_LT_DT
#undef ISSM_LT
#undef ISSM_LT_ONE
#undef ISSM_LT_FORM
  return (int)hipGetLastError();
}

}  // namespace issm
