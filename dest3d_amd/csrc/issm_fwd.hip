// Forward kernels of the ISSM chunked scan for gfx950.
//
//   k_chunk_local   dt transform + cumsum, chunk-local end states S_c and the intra-chunk
//                   matrix M_c = "C.A.B^T" in one pass over dt, in the form below; calls without
//                   packed sequences take k_local_tile (issm_fwd_tile.hip) from four state columns on
//   k_chunk_scan    y = (C*exp(cs)) H^T + tril(M) x + D x, optional gate
//
// The decay exp(cs[l]-cs[s]) sits inside the contraction over the state index n, so
// M = sum_n C[l,n] B[s,n] dt'[s,n] exp(cs[l,n]-cs[s,n]) is not a plain GEMM.  It is
// evaluated exactly on the matrix cores by a binary hierarchy over the rows of a chunk:
// a pair (l > s) belongs to level w = highest set bit of (l xor s); at that level both
// rows sit in the same aligned block of 2w rows, s in its lower half, l in its upper half,
// and with r = last row of the lower half
//        exp(cs[l]-cs[s]) = exp(cs[l]-cs[r]) * exp(cs[r]-cs[s]).
// dt' >= 0 makes cs monotone in l for every n, so both factors lie between 1 and the
// product: nothing overflows that the exact value would not.  Level w therefore is an
// ordinary product Cw . Bw^T of rescaled operands, restricted to its blocks.  Levels 32 and 16
// are products of whole 16-row tiles, levels 8 and 4 live inside a diagonal tile (there one
// operand t = C exp2(cs - ref) on upper rows, Bd exp2(ref - cs) on lower rows serves as both
// factors: t . t^T holds the wanted entries where the row is upper and the column lower), and
// the pairs of levels 2, 1 and the diagonal belong to a single lane of the column-lane layout,
// which evaluates them directly with one exp2 per pair.
#include "issm_dev.h"
#include "issm_fwd_local.h"

namespace issm {

template <int PT, bool IOB, bool DTB, bool FULL>
__global__ __launch_bounds__(NTHREADS, 2) void k_chunk_local(KP p, float* __restrict__ states, float* __restrict__ cs_last, float* __restrict__ cabt) {
  k_chunk_local_body<PT, IOB, DTB, FULL>(p, states, cs_last, cabt);
}

// ------------------------------------------------------------------ chunk scan
// BF (bf16 inputs): the operands of the product over the state index are bf16 tiles read as matrix fragments of 8
// adjacent columns; fp32 inputs: (hi, lo) pairs of such tiles from two head tiles on, fp32 tiles for one.
#ifndef SCAN_SPLIT_FROM
#define SCAN_SPLIT_FROM 2
#endif
template <int PT, bool BF, int NG>
struct FwdScanSmem {
  static constexpr int LDK = NS + 8;  // row stride of the bf16 tiles
  // fp32 inputs: the product over the state index on (hi, lo) bf16 tiles, hi.hi + hi.lo + lo.hi, instead of fp32
  // matrix instructions.  An fp32 matrix instruction takes the vector ALU's issue slots (the two never overlap on this
  // chip): they were 31 % of the kernel's issue cycles beside 46 % of vector work with two head tiles, 46 % beside
  // 39 % with four.  Three bf16 instructions per product take a fifth of that and run beside the vector ALU; the
  // splitting adds a quarter to the vector work.  (SCAN_SPLIT_FROM: head tiles from which this form is used.)
  static constexpr bool SPL = !BF && PT >= SCAN_SPLIT_FROM;
  static constexpr bool B16 = BF || SPL;
  static constexpr int NH = SPL ? 2 : 1;
  float xs[RowTile<PT>::SIZE];                                  // x [s][p]
  static constexpr int CT = NH * CS * (B16 ? LDK : LDN), HS = NH * PT * 16 * (B16 ? LDK : LDN);
  typedef typename std::conditional<B16, uint16_t, float>::type Op;
  alignas(16) Op ct[NG * CT];  // C * exp2(cs) [l][n], a tile a group of waves
  Op hs[NG * HS];              // H [p][n]
  static_assert(NG == 1 || NG * CT * sizeof(Op) >= PT * NTHREADS * sizeof(f4), "the second group's sums take the place of the tiles");
};
// a (16 PT x 64) slab of fp32 values (layout of pn_load) rounded to bf16 into LDS dst[p][col], row stride LD
template <int PT, int LD>
__device__ __forceinline__ void pn_store_bf(const PnRegs<PT>& r, uint16_t* dst, int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
#pragma unroll
  for (int i = 0; i < R::CNT; ++i) {
    const int e = tid + i * NTHREADS, pp = e / R::Q, c4 = (e % R::Q) * 4;
    if (e < R::TOT) *(uint2*)(dst + pp * LD + c4) = make_uint2(pack_bf16(r.v[i][0], r.v[i][1]), pack_bf16(r.v[i][2], r.v[i][3]));
  }
}
// the same slab as (hi, lo) bf16 pairs
template <int PT, int LD>
__device__ __forceinline__ void pn_store_split(const PnRegs<PT>& r, uint16_t* hi, uint16_t* lo, int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
#pragma unroll
  for (int i = 0; i < R::CNT; ++i) {
    const int e = tid + i * NTHREADS, pp = e / R::Q, c4 = (e % R::Q) * 4;
    const float w[4] = {r.v[i][0], r.v[i][1], r.v[i][2], r.v[i][3]};
    bf4 h, l;
    split4(w, h, l);
    if (e < R::TOT) {
      *(bf4*)(hi + pp * LD + c4) = h;
      *(bf4*)(lo + pp * LD + c4) = l;
    }
  }
}
// the lane's 16 values of one column -> column `col` of a [64][LD] bf16 tile
template <int LD>
__device__ __forceinline__ void col_store_bf(const float (&v)[16], uint16_t* dst, int g4, int col) {
#pragma unroll
  for (int k = 0; k < 16; k += 2) {
    const unsigned h2 = pack_bf16(v[k], v[k + 1]);
    dst[lane_row(k, g4) * LD + col] = (uint16_t)h2;
    dst[lane_row(k + 1, g4) * LD + col] = (uint16_t)(h2 >> 16);
  }
}

// NG: groups of four waves.  Two take every second slice of the states each where the grid gives a CU no second workgroup to run
// beside this one; the second adds M x.
template <int PT, bool IOB, bool DTB, bool FULL, int NG>
__device__ __forceinline__ void k_chunk_scan_body(const KP& p, const float* __restrict__ states, const float* __restrict__ cabt, float* __restrict__ out_x) {
  warm_args();
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef FwdScanSmem<PT, IOB, NG> SM;
  SM& s = *reinterpret_cast<SM*>(smem_raw);
  typedef RowTile<PT> XT;
  constexpr int LDX = XT::LD, LDK = SM::LDK;
  constexpr int STEP = NG * NS;
  const int tid = NG > 1 ? threadIdx.x & (NTHREADS - 1) : threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = NG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NTHREADS) : 0;
  typename SM::Op *ct = s.ct + grp * SM::CT, *hs = s.hs + grp * SM::HS;
  const int cm = lane & 15, g4 = lane >> 4;
  const Unit u = decode_unit(p, xcd_remap(blockIdx.x, gridDim.x));
  const float* hsrc = states + st_off(p, u.bt, u.c, u.h);

  int n = grp * NS + wave * 16 + cm;
  bool vn = FULL || n < p.N;
  RowMap rm;
  Coef cf;
  rm = make_rowmap<FULL>(p, u, g4, grp * NS);
  float raw[16], cv[16];
  PnRegs<PT> hv;
  lane_load_ln<DTB>(p.dt, u.b, u.h, n, vn, g4, rm, raw);
  cf = lane_coef(p, u.h, n, vn);
  lane_load_ln<IOB>(p.Cm[u.dir], u.b, u.g, n, vn, g4, rm, cv);
  pn_load<PT, FULL>(p, hsrc, grp * NS, hv, tid);
  if (grp == NG - 1) {
    float xv[CS * PT * 16 / NTHREADS];
    lp_load<IOB, PT, FULL>(p, u, p.x[u.dir], xv, tid);
    lp_store<PT>(xv, s.xs, tid);
  }
  f4 acc[PT];
#pragma unroll
  for (int pt = 0; pt < PT; ++pt) acc[pt] = (f4){0, 0, 0, 0};

  for (int m0 = 0; m0 < p.N; m0 += STEP) {
    const int n0 = m0 + grp * NS;
    const bool mine = NG == 1 || n0 < p.N;   // uniform
    if (mine) {
      float dtp[16], cs[16], dummy[16];
      lane_prep<false>(p, cf, vn, cm, g4, rm, raw, dtp, cs, dummy);
      if constexpr (IOB) {
        float ctv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) ctv[k] = cv[k] * ex2(cs[k]);
        col_store_bf<LDK>(ctv, ct, g4, wave * 16 + cm);
      } else if constexpr (SM::SPL) {
        float ctv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) ctv[k] = cv[k] * ex2(cs[k]);
        op_store<LDK, true>(ctv, ct, ct + CS * LDK, g4, wave * 16 + cm);
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) ct[lane_row(k, g4) * LDN + wave * 16 + cm] = cv[k] * ex2(cs[k]);
      }
      if constexpr (!FULL) pn_edge<PT>(p, n0, hv, tid);
      if constexpr (IOB) pn_store_bf<PT, LDK>(hv, hs, tid);
      else if constexpr (SM::SPL) pn_store_split<PT, LDK>(hv, hs, hs + PT * 16 * LDK, tid);
      else pn_store<PT>(hv, hs, tid);
    }
    if (n0 + STEP < p.N) {
      n = n0 + STEP + wave * 16 + cm;
      vn = FULL || n < p.N;
      rm = make_rowmap<FULL>(p, u, g4, n0 + STEP);
      lane_load_ln<DTB>(p.dt, u.b, u.h, n, vn, g4, rm, raw);
      cf = lane_coef(p, u.h, n, vn);
      lane_load_ln<IOB>(p.Cm[u.dir], u.b, u.g, n, vn, g4, rm, cv);
      pn_load<PT, FULL>(p, hsrc, n0 + STEP, hv, tid);
    }
    __syncthreads();
    // y[l][p] += sum_n Ct[l][n] H[p][n]; wave owns 16 rows
    if (!mine) {
    } else if constexpr (IOB) {
      // bf16 inputs: one rounding of C exp(cs) and of the entry state to bf16 (the reference stores the entry states
      // in the input dtype and casts its dot operands, issm_combined.py:87, issm_chunk_scan.py:149-190)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf8 a = op_frag<LDK>(ct, wave * 16 + cm, g4, t);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) acc[pt] = mfma_bf(a, op_frag<LDK>(hs, pt * 16 + cm, g4, t), acc[pt]);
      }
    } else if constexpr (SM::SPL) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf8 ah = op_frag<LDK>(ct, wave * 16 + cm, g4, t), al = op_frag<LDK>(ct + CS * LDK, wave * 16 + cm, g4, t);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
          acc[pt] = mfma_split(ah, al, op_frag<LDK>(hs, pt * 16 + cm, g4, t),
                               op_frag<LDK>(hs + PT * 16 * LDK, pt * 16 + cm, g4, t), acc[pt]);
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < NS; kb += 16)
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) mma16_mm(acc[pt], ct, LDN, wave * 16, hs, LDN, pt * 16, kb, lane);
    }
    __syncthreads();
  }
  // Requested here and not with the first step's operands: over the loop its 16 registers pushed 8 dwords a lane to scratch at 128
  // registers, or kept a fourth workgroup off the CU.
  // M of this wave's 16 rows goes straight into matrix-operand registers (lane (row cm, group g4) holds columns
  // 16 kb + 4 g4 .. + 3 of the blocks kb <= wave, the upper triangle of the diagonal block zeroed): no LDS tile, which
  // lets a fourth workgroup live on the CU
  if (grp == NG - 1) {
    f4 mf[4];
    {
      const float* mrow = cabt + sq_off(p, u.bt, u.c, u.h) + (wave * 16 + cm) * CS + 4 * g4;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) mf[kb] = *(const f4*)(mrow + 16 * min(kb, wave));  // no branch between the loads
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (kb > wave || (kb == wave && 4 * g4 + j > cm)) mf[kb][j] = 0.0f;
    }
    // y[l][p] += sum_{s<=l} M[l][s] x[s][p]; rows of this wave only need s < 16(wave+1)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      if (kb <= wave) {  // uniform
        // the lane's four M values and four x values are the operands of one K = 16 bf16 instruction as they stand
        // (k-slot j of lane group g4 <-> row 16 kb + 4 g4 + j), M as a (hi, lo) pair and, for fp32 inputs, x too
        const float mw[4] = {mf[kb][0], mf[kb][1], mf[kb][2], mf[kb][3]};
        bf4 ah, al;
        split4(mw, ah, al);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
          const float* bp = s.xs + XT::at(16 * kb + 4 * g4, pt * 16 + cm);
          const float xw[4] = {bp[0], bp[LDX], bp[2 * LDX], bp[3 * LDX]};
          bf4 bh, bl;
          split4(xw, bh, bl);
          acc[pt] = mfma_bf16k(al, bh, acc[pt]);
          if constexpr (!IOB) acc[pt] = mfma_bf16k(ah, bl, acc[pt]);  // (bf16 inputs: x is exact, its lo part zero)
          acc[pt] = mfma_bf16k(ah, bh, acc[pt]);
        }
      }
  }
  if constexpr (NG > 1) {
    f4* part = (f4*)s.ct;
    if (grp) {
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) part[pt * NTHREADS + tid] = acc[pt];
    }
    __syncthreads();
    if (grp) return;
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) acc[pt] += part[pt * NTHREADS + tid];
  }

  const TensorD& to = p.out[u.dir];
  const TensorD& tz = p.z[u.dir];
#pragma unroll
  for (int pt = 0; pt < PT; ++pt) {
    int off[4];
    float v[4];
    // the skip coefficient of the lane's column, read once and without a lane-dependent branch (absent columns read
    // the head's last one; their results are not stored)
    float dcoef = 0.0f;
    if (p.D) dcoef = (p.flags & F_D_HDIM) ? p.D[u.h * p.P + min(pt * 16 + cm, p.P - 1)] : p.D[u.h];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int l = wave * 16 + 4 * g4 + r, pp = pt * 16 + cm;
      const int tt = u.c * CS + l;
      const bool ok = tt < p.L && pp < p.P;
      const int pr = ok ? phys_row(p, u.dir, tt) : 0;
      v[r] = fmaf(dcoef, s.xs[XT::at(l, pp)], acc[pt][r]);
      if (tz.ptr && ok) {
        if (out_x) out_x[(((long)u.bt * p.L + pr) * p.H + u.h) * p.P + pp] = v[r];
        const float zz = ldv(tz.ptr, (long)u.b * tz.s0 + (long)pr * tz.s1 + (long)u.h * tz.s2 + pp, p.io_dt);
        v[r] *= zz * sigmoidf_(zz);
      }
      off[r] = ok ? pr * (int)to.s1 + pp : -1;
    }
    gstore<IOB, 4>(const_cast<void*>(to.ptr), (long)u.b * to.s0 + (long)u.h * to.s2, off, v);
  }
}
// two head tiles, fp32 inputs or edges: 128 registers, so that a fourth workgroup lives on the CU (52 -> 48.5 us)
template <int PT, bool IOB, bool DTB, bool FULL, int NG>
__global__ __launch_bounds__(NG * NTHREADS, (PT <= 2 && NG == 1 && (!IOB || !FULL)) ? 4 : 1) void k_chunk_scan(KP p, const float* __restrict__ states, const float* __restrict__ cabt, float* __restrict__ out_x) {
  k_chunk_scan_body<PT, IOB, DTB, FULL, NG>(p, states, cabt, out_x);
}

// ------------------------------------------------------------------- launchers
template <typename K>
static int set_lds(K kernel, size_t bytes) {   // (up to 64 KB needs no asking)
  return bytes > 64 * 1024 ? (int)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) : 0;
}

bool local_tile_available(const KP& p, const float* states, const float* cabt);
int launch_local_tile(const KP& p, float* states, float* cs_last, float* cabt, bool any, hipStream_t st);

// The row-lane kernel takes what it can (it falls back to the level-hierarchy body itself for the chunks outside its
// range or, any, evaluates their bf16 tiles in place); packed sequences and calls that want one output only go to the level-hierarchy kernel.
int launch_chunk_local(const KP& p, float* states, float* cs_last, float* cabt, bool any, hipStream_t st) {
  if (local_tile_available(p, states, cabt)) return launch_local_tile(p, states, cs_last, cabt, any, st);
  const int units = p.B * p.ndir * p.nc * p.H;
  ISSM_DISPATCH(p, {
    const size_t sm = sizeof(FwdLocalSmem<PT_, !IOB_>);
    constexpr auto kern = &k_chunk_local<PT_, IOB_, DTB_, FULL_>;
    if (int e = set_lds(kern, sm)) return e;
    hipLaunchKernelGGL(kern, dim3(units), dim3(NTHREADS), sm, st, p, states, cs_last, cabt);
  });
  return (int)hipGetLastError();
}

int launch_chunk_scan(const KP& p, const float* states, const float* cabt, float* out_x, hipStream_t st) {
  const int units = p.B * p.ndir * p.nc * p.H;
  ISSM_DISPATCH(p, {
    if (two_groups(units, p.N)) {
      const size_t sm = sizeof(FwdScanSmem<PT_, IOB_, 2>);
      constexpr auto kern = &k_chunk_scan<PT_, IOB_, DTB_, FULL_, 2>;
      if (int e = set_lds(kern, sm)) return e;
      hipLaunchKernelGGL(kern, dim3(units), dim3(2 * NTHREADS), sm, st, p, states, cabt, out_x);
    } else {
      const size_t sm = sizeof(FwdScanSmem<PT_, IOB_, 1>);
      constexpr auto kern = &k_chunk_scan<PT_, IOB_, DTB_, FULL_, 1>;
      if (int e = set_lds(kern, sm)) return e;
      hipLaunchKernelGGL(kern, dim3(units), dim3(NTHREADS), sm, st, p, states, cabt, out_x);
    }
  });
  return (int)hipGetLastError();
}

}  // namespace issm
