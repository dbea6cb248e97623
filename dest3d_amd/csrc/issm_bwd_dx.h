// dx of a chunk and head, and its partial sums of dD: the body of k_bwd_dx (issm_bwd.hip), which k_bwd_tile (issm_bwd_tile.hip) takes
// into its launch where both leave most of the chip idle.
#pragma once
#include "issm_dev.h"

namespace issm {

// BF (bf16 inputs): the operands of the product over the state index are bf16 tiles read as matrix fragments of 8
// adjacent columns; fp32 inputs: (hi, lo) pairs of such tiles from two head tiles on, fp32 tiles for one.  `prod` (the
// dy * x products of the skip gradient) is its own small tile for bf16 inputs.
#ifndef DX_SPLIT_FROM
#define DX_SPLIT_FROM 2
#endif
template <int PT, bool BF, int NG>
struct BwdDxSmem {
  static constexpr int LDK = NS + 8;
  // fp32 inputs: the product over the state index on (hi, lo) bf16 tiles, hi.hi + hi.lo + lo.hi, instead of fp32
  // matrix instructions, which take the vector ALU's issue slots (28 - 45 % of this kernel's cycles, never beside its
  // vector work); the bf16 instructions run beside it.  (DX_SPLIT_FROM: head tiles from which this form is used.)
  static constexpr bool SPL = !BF && PT >= DX_SPLIT_FROM;
  static constexpr bool B16 = BF || SPL;
  static constexpr int NH = SPL ? 2 : 1;
  float dys[RowTile<PT>::SIZE];
  static constexpr int BT = NH * CS * (B16 ? LDK : LDN), DS = NH * PT * 16 * (B16 ? LDK : LDN);
  typedef typename std::conditional<B16, uint16_t, float>::type Op;
  alignas(16) Op bt[NG * BT];  // B dt' exp2(last - cs) [m][n], a tile a group of waves
  Op dss[NG * DS];             // dS [p][n]
  static_assert(NG == 1 || NG * BT * sizeof(Op) >= PT * NTHREADS * sizeof(f4), "the second group's sums take the place of the tiles");
  // dy * x, in the place of `bt` and `dss` once their product is done
  static constexpr int LDPROD = B16 ? PT * 16 + 4 : LDN;
  __device__ __forceinline__ float* prod() { return reinterpret_cast<float*>(bt); }
  static_assert(sizeof(bt) % 16 == 0 && sizeof(bt) + sizeof(dss) >= sizeof(float) * CS * LDPROD, "dy * x fits");
};
// a (16 PT x 64) slab of fp32 values as (hi, lo) bf16 pairs into LDS hi / lo [p][col], row stride LD
template <int PT, int LD>
__device__ __forceinline__ void pn_store_hl(const PnRegs<PT>& r, uint16_t* hi, uint16_t* lo, int tid = threadIdx.x) {
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
template <int PT, int LD>
__device__ __forceinline__ void pn_store_bf16(const PnRegs<PT>& r, uint16_t* dst, int tid = threadIdx.x) {
  typedef PnRegs<PT> R;
#pragma unroll
  for (int i = 0; i < R::CNT; ++i) {
    const int e = tid + i * NTHREADS, pp = e / R::Q, c4 = (e % R::Q) * 4;
    if (e < R::TOT) *(uint2*)(dst + pp * LD + c4) = make_uint2(pack_bf16(r.v[i][0], r.v[i][1]), pack_bf16(r.v[i][2], r.v[i][3]));
  }
}
template <int LD>
__device__ __forceinline__ bf8 frag8(const uint16_t* tile, int row, int g4, int t) {
  return *(const bf8*)(tile + row * LD + 32 * t + 8 * g4);
}

// partD: (Bt*nc*H, P) per-unit sums over rows of dy*x
// NG: groups of four waves, as in k_chunk_scan.
template <int PT, bool IOB, bool DTB, bool FULL, int NG>
__device__ __forceinline__ void k_bwd_dx_body(const KP& p, int block, int blocks, const float* __restrict__ dy_ws, const float* __restrict__ dstates, const float* __restrict__ cabt, float* __restrict__ partD) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef BwdDxSmem<PT, IOB, NG> SM;
  SM& s = *reinterpret_cast<SM*>(smem_raw);
  typedef RowTile<PT> YT;
  constexpr int LDY = YT::LD, LDK = SM::LDK, LDPR = SM::LDPROD;
  constexpr int STEP = NG * NS;
  const int tid = NG > 1 ? threadIdx.x & (NTHREADS - 1) : threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = NG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NTHREADS) : 0;
  typename SM::Op *bt = s.bt + grp * SM::BT, *dss = s.dss + grp * SM::DS;
  const int cm = lane & 15, g4 = lane >> 4;
  warm_args();
  const Unit u = decode_unit(p, xcd_remap(block, blocks));
  const float* ds = dstates + dst_off(p, u.bt, u.c, u.h);

  int n = grp * NS + wave * 16 + cm;
  bool vn = FULL || n < p.N;
  RowMap rm;
  Coef cf;
  rm = make_rowmap<FULL>(p, u, g4, grp * NS);
  float raw[16], bv[16];
  PnRegs<PT> sv;
  lane_load_ln<DTB>(p.dt, u.b, u.h, n, vn, g4, rm, raw);
  cf = lane_coef(p, u.h, n, vn);
  lane_load_ln<IOB>(p.Bm[u.dir], u.b, u.g, n, vn, g4, rm, bv);
  pn_load<PT, FULL>(p, ds, grp * NS, sv, tid);
  if (grp == NG - 1) {
    float dv[CS * PT * 16 / NTHREADS];
    dy_load<IOB, PT, FULL>(p, u, dy_ws, dv, tid);
    lp_store<PT>(dv, s.dys, tid);
  }
  f4 acc[PT];
#pragma unroll
  for (int pt = 0; pt < PT; ++pt) acc[pt] = (f4){0, 0, 0, 0};

  for (int m0 = 0; m0 < p.N; m0 += STEP) {
    const int n0 = m0 + grp * NS;
    const bool mine = NG == 1 || n0 < p.N;   // uniform
    if (mine) {
      float dtp[16], cs[16], dummy[16];
      const float last = lane_prep<false>(p, cf, vn, cm, g4, rm, raw, dtp, cs, dummy);
      if constexpr (IOB) {
        float btv[16];
#pragma unroll
        for (int k = 0; k < 16; k += 2) {
          btv[k] = bv[k] * dtp[k] * ex2(last - cs[k]);
          btv[k + 1] = bv[k + 1] * dtp[k + 1] * ex2(last - cs[k + 1]);
          const unsigned h2 = pack_bf16(btv[k], btv[k + 1]);
          bt[lane_row(k, g4) * LDK + wave * 16 + cm] = (uint16_t)h2;
          bt[lane_row(k + 1, g4) * LDK + wave * 16 + cm] = (uint16_t)(h2 >> 16);
        }
      } else if constexpr (SM::SPL) {
#pragma unroll
        for (int k = 0; k < 16; k += 2) {
          const float b0 = bv[k] * dtp[k] * ex2(last - cs[k]), b1 = bv[k + 1] * dtp[k + 1] * ex2(last - cs[k + 1]);
          const unsigned h2 = pack_bf16(b0, b1);
          const unsigned l2 = pack_bf16(b0 - __uint_as_float(h2 << 16), b1 - __uint_as_float(h2 & 0xffff0000u));
          const int o0 = lane_row(k, g4) * LDK + wave * 16 + cm, o1 = lane_row(k + 1, g4) * LDK + wave * 16 + cm;
          bt[o0] = (uint16_t)h2;
          bt[o1] = (uint16_t)(h2 >> 16);
          bt[CS * LDK + o0] = (uint16_t)l2;
          bt[CS * LDK + o1] = (uint16_t)(l2 >> 16);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k)
          bt[lane_row(k, g4) * LDN + wave * 16 + cm] = bv[k] * dtp[k] * ex2(last - cs[k]);
      }
      if constexpr (!FULL) pn_edge<PT>(p, n0, sv, tid);
      if constexpr (IOB) pn_store_bf16<PT, LDK>(sv, dss, tid);
      else if constexpr (SM::SPL) pn_store_hl<PT, LDK>(sv, dss, dss + PT * 16 * LDK, tid);
      else pn_store<PT>(sv, dss, tid);
    }
    if (n0 + STEP < p.N) {
      n = n0 + STEP + wave * 16 + cm;
      vn = FULL || n < p.N;
      rm = make_rowmap<FULL>(p, u, g4, n0 + STEP);
      lane_load_ln<DTB>(p.dt, u.b, u.h, n, vn, g4, rm, raw);
      cf = lane_coef(p, u.h, n, vn);
      lane_load_ln<IOB>(p.Bm[u.dir], u.b, u.g, n, vn, g4, rm, bv);
      pn_load<PT, FULL>(p, ds, n0 + STEP, sv, tid);
    }
    __syncthreads();
    if (!mine) {
    } else if constexpr (IOB) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf8 a = frag8<LDK>(bt, wave * 16 + cm, g4, t);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) acc[pt] = mfma_bf(a, frag8<LDK>(dss, pt * 16 + cm, g4, t), acc[pt]);
      }
    } else if constexpr (SM::SPL) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf8 ah = frag8<LDK>(bt, wave * 16 + cm, g4, t), al = frag8<LDK>(bt + CS * LDK, wave * 16 + cm, g4, t);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
          acc[pt] = mfma_split(ah, al, frag8<LDK>(dss, pt * 16 + cm, g4, t),
                               frag8<LDK>(dss + PT * 16 * LDK, pt * 16 + cm, g4, t), acc[pt]);
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < NS; kb += 16)
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) mma16_mm(acc[pt], bt, LDN, wave * 16, dss, LDN, pt * 16, kb, lane);
    }
    __syncthreads();
  }
  // (requested behind the loop, as in k_chunk_scan: 44 bytes a lane of scratch at 128 registers otherwise.  Four head tiles, fp32,
  // incomplete, take 36 bytes the other way round, and the same time, 8 x 1000 tokens, 8 heads x 64, 250 states: 98.2 us both, one
  // direction 55.3 and 56.2 with M in front)
  // M^T of this wave's 16 columns goes straight into matrix-operand registers (lane (column cm, group g4) holds
  // rows 16 kb + 4 g4 .. + 3 of the blocks kb >= wave, the upper triangle of the diagonal block zeroed): no LDS tile,
  // which lets a fourth workgroup live on the CU
  if (grp == NG - 1) {
    float mf[4][4];
    {
      const float* mcol = cabt + sq_off(p, u.bt, u.c, u.h) + (4 * g4) * CS + wave * 16 + cm;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) mf[kb][j] = mcol[(16 * max(kb, wave) + j) * CS];  // no branch between the loads
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (kb < wave || (kb == wave && cm > 4 * g4 + j)) mf[kb][j] = 0.0f;
    }
    // dx[m][p] += sum_{l>=m} M[l][m] dy[l][p]
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      if (kb >= wave) {  // uniform
        // the lane's four M values and four dy values are the operands of one K = 16 bf16 instruction as they stand
        // (k-slot j of lane group g4 <-> row 16 kb + 4 g4 + j), both as (hi, lo) pairs
        bf4 ah, al;
        split4(mf[kb], ah, al);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
          const float* bp = s.dys + YT::at(16 * kb + 4 * g4, pt * 16 + cm);
          const float yw[4] = {bp[0], bp[LDY], bp[2 * LDY], bp[3 * LDY]};
          bf4 bh, bl;
          split4(yw, bh, bl);
          acc[pt] = mfma_bf16k(al, bh, acc[pt]);
          acc[pt] = mfma_bf16k(ah, bl, acc[pt]);  // (also for bf16 inputs: a gated dy is an fp32 product)
          acc[pt] = mfma_bf16k(ah, bh, acc[pt]);
        }
      }
  }
  if constexpr (NG > 1) {
    f4* part = (f4*)s.bt;
    if (grp) {
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) part[pt * NTHREADS + tid] = acc[pt];
    }
    __syncthreads();
    if (grp) return;
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) acc[pt] += part[pt * NTHREADS + tid];
    __syncthreads();   // dy * x goes where these were
  }

  const TensorD& tx = p.x[u.dir];
  const TensorD& tdx = p.dx[u.dir];
  float* prod = s.prod();  // [64][LDPR]
#pragma unroll
  for (int pt = 0; pt < PT; ++pt) {
    int ox[4], odx[4];
    float xv[4], v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int l = wave * 16 + 4 * g4 + r, pp = pt * 16 + cm, tt = u.c * CS + l;
      const bool ok = tt < p.L && pp < p.P;
      const int pr = ok ? phys_row(p, u.dir, tt) : 0;
      ox[r] = (ok && p.D) ? pr * (int)tx.s1 + pp : -1;
      odx[r] = (ok && tdx.ptr) ? pr * (int)tdx.s1 + pp : -1;
    }
    gload<IOB, 4>(tx.ptr, (long)u.b * tx.s0 + (long)u.h * tx.s2, ox, xv);
    float dcoef = 0.0f;  // skip coefficient of the lane's column, read once
    if (p.D) dcoef = (p.flags & F_D_HDIM) ? p.D[u.h * p.P + min(pt * 16 + cm, p.P - 1)] : p.D[u.h];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int l = wave * 16 + 4 * g4 + r, pp = pt * 16 + cm;
      const float dyv = s.dys[YT::at(l, pp)];
      v[r] = fmaf(dcoef, dyv, acc[pt][r]);
      prod[l * LDPR + pp] = dyv * xv[r];
    }
    gstore<IOB, 4>(const_cast<void*>(tdx.ptr), (long)u.b * tdx.s0 + (long)u.h * tdx.s2, odx, v);
  }
  if (p.D && partD) {
    __syncthreads();
    if (tid < PT * 16) {
      float sum = 0.0f;
      for (int l = 0; l < CS; ++l) sum += prod[l * LDPR + tid];
      if (tid < p.P) partD[(((long)u.bt * p.nc + u.c) * p.H + u.h) * p.P + tid] = sum;
    }
  }
}

}  // namespace issm
