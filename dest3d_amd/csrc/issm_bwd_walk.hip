// Backward pass over the chunk states in one kernel (gfx950): dH_c = dy^T (C exp(cs)), the reverse recurrence over the chunks
// and the matrix dM, for calls whose sequences and column slices fill the chip or that have few chunks (bwd_walks, issm_abi.hip).
//
// Workgroup = (batch and direction, head, 64 state columns), walking the chunks from the last to the first.  dH contracts over
// the rows of a chunk and the recurrence is element-wise, so neither needs another workgroup's columns: the lane that owns
// column n and rows p = 16 pt + 4 g4 + r of the state keeps them in the accumulator of the matrix instruction that adds the next
// dH,
//     dS_c = carry (stored),   carry = exp(chunk total) carry + dy^T (C exp(cs)).
// As two kernels (k_bwd_dstates, k_state_pass) the same work writes dH and reads it back, 8 P N bytes a chunk and head.
// Every operand of chunk c - 1 is requested while chunk c is computed; dy's tile, which the four waves share, is staged
// transposed in two LDS buffers used in turn: one barrier a chunk.
//
// dM = tril(dy x^T) needs no state column: workgroups behind the walks in the same launch take it, one a chunk and head, and run
// where the walks leave room on the CUs (the walks wait for one another's latencies: dealt to their waves instead, dM's ten blocks
// held every chunk up, by 14 us at the first size below).  It leaves as the symmetric bf16 matrix (and, fp32 inputs, the
// second one with what the first left) that k_bwd_dstates describes: the same products in the same order.
//
// Both kernels -> this one: 8 x 1024 tokens, both directions, 8 heads x 32, 256 states 74 -> 61 us fp32, 62 -> 46 bf16 (285 MB
// fp32: 4.7 TB/s); heads of 36, bf16 68 -> 51; 4 x 2048, 16 heads x 64, 512 states fp32 540 -> 350, bf16 485 -> 271.
#include "issm_dev.h"

namespace issm {

template <int PT, bool BF>
struct BwdWalkSmem {
  static constexpr int LDT = CS + 8;   // dy tile transposed, [p][l]
  uint16_t hi[2][PT * 16 * LDT];
  uint16_t lo[2][BF ? 8 : PT * 16 * LDT];
};

// What both kinds of workgroup read of a (B, L, H, P) tensor: four elements of row l (scan order) of chunk c from column p4 on;
// where they do not exist, four that do.
template <bool BF, bool FULL>
struct RowsOf {
  typedef typename std::conditional<BF, uint16_t, float>::type T;
  typedef typename std::conditional<BF, uint2, f4>::type V;
  const T* q;
  int s1, t0, sgn, L, P;
  __device__ __forceinline__ RowsOf(const KP& p, const TensorD& t, const Unit& u)
      : q((const T*)t.ptr + ((long)u.b * t.s0 + (long)u.h * t.s2)), s1((int)t.s1), t0(u.dir ? p.L - 1 : 0), sgn(u.dir ? -1 : 1), L(p.L), P(p.P) {}
  __device__ __forceinline__ bool has(int c, int l, int p4) const { return p4 < P && (FULL || l < L - c * CS); }
  __device__ __forceinline__ V get(int c, int l, int p4) const { return *(const V*)(q + (has(c, l, p4) ? (t0 + sgn * (c * CS + l)) * s1 + p4 : 0)); }
};
__device__ __forceinline__ TensorD dy_of(const KP& p, const Unit& u, const float* dy_ws) {
  TensorD t = p.dout[u.dir];
  if (dy_ws) {   // gated: the fp32 (Bt, L, H, P) copy
    t.ptr = dy_ws + (long)(u.bt - u.b) * p.L * p.H * p.P;
    t.s0 = (long)p.L * p.H * p.P;
    t.s1 = (long)p.H * p.P;
    t.s2 = p.P;
  }
  return t;
}

// dM of unit `id`: wave w takes the blocks (w, j <= w).
template <int PT, bool BF, bool FULL>
__device__ __forceinline__ void dm_unit(const KP& p, const float* dy_ws, float* dm, int id) {
  constexpr int KT = (PT + 1) / 2;
  typedef RowsOf<BF, FULL> Rows;
  typedef typename Rows::V V;
  const int lane = threadIdx.x & 63, cm = lane & 15, g4 = lane >> 4;
  const int i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Unit u = decode_unit(p, id);
  const Rows ry(p, dy_of(p, u, dy_ws), u), rx(p, p.x[u.dir], u);
  // the lane's operands of a 16-row tile: row 16 tile + cm, k-slots as split_frag has them
  struct Op {
    bf8 h[KT], l[KT];
  };
  auto operand = [&](const Rows& r, int tile) -> Op {
    V v[KT][2];
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e) v[t][e] = r.get(u.c, 16 * tile + cm, 32 * t + 16 * e + 4 * g4);
    Op o;
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const bool a = r.has(u.c, 16 * tile + cm, 32 * t + 4 * g4), b = r.has(u.c, 16 * tile + cm, 32 * t + 16 + 4 * g4);
      if constexpr (BF) {
        const uint2 z = make_uint2(0u, 0u), v0 = a ? v[t][0] : z, v1 = b ? v[t][1] : z;
        o.h[t] = __builtin_bit_cast(bf8, make_uint4(v0.x, v0.y, v1.x, v1.y));
      } else {
        float w[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          w[k] = a ? v[t][0][k] : 0.0f;
          w[4 + k] = b ? v[t][1][k] : 0.0f;
        }
        split8(w, o.h[t], o.l[t]);
      }
    }
    return o;
  };
  const Op y = operand(ry, i);
  uint16_t* m = reinterpret_cast<uint16_t*>(dm + sq_off(p, u.bt, u.c, u.h));
  for (int j = 0; j <= i; ++j) {
    const Op x = operand(rx, j);
    // the block both ways round, so that it and its mirror image leave in 8-byte pieces of rows: acc row 4 g4 + r of dy, column cm
    // of x; tra the other way round, the same products in the same order
    f4 acc = {0, 0, 0, 0}, tra = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      if constexpr (!BF) {
        acc = mfma_bf(y.l[t], x.h[t], acc);
        acc = mfma_bf(y.h[t], x.l[t], acc);
        tra = mfma_bf(x.h[t], y.l[t], tra);
        tra = mfma_bf(x.l[t], y.h[t], tra);
      }
      acc = mfma_bf(y.h[t], x.h[t], acc);
      tra = mfma_bf(x.h[t], y.h[t], tra);
    }
    if (i == j) {   // uniform; what lies above the diagonal is what lies below it
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = tra[r] = cm >= 4 * g4 + r ? tra[r] : acc[r];
    }
    const int at_acc = (16 * j + cm) * CS + 16 * i + 4 * g4, at_tra = (16 * i + cm) * CS + 16 * j + 4 * g4;
#pragma unroll
    for (int h = 0; h < (BF ? 1 : 2); ++h) {
      const uint2 wa = make_uint2(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]));
      const uint2 wt = make_uint2(pack_bf16(tra[0], tra[1]), pack_bf16(tra[2], tra[3]));
      *(uint2*)(m + h * CS * CS + at_acc) = wa;
      *(uint2*)(m + h * CS * CS + at_tra) = wt;
      if (h == 0 && !BF) {
        const unsigned ua[2] = {wa.x, wa.y}, ut[2] = {wt.x, wt.y};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[r] -= __uint_as_float((r & 1) ? ua[r >> 1] & 0xffff0000u : ua[r >> 1] << 16);
          tra[r] -= __uint_as_float((r & 1) ? ut[r >> 1] & 0xffff0000u : ut[r >> 1] << 16);
        }
      }
    }
  }
}

// PT, BF, FULL as in the other kernels; x / B / C / dt of one type, rows of x and dy in accesses of four elements (the host checks).
// The first `walks` workgroups walk, the others are dM's.
template <int PT, bool BF, bool FULL>
__global__ __launch_bounds__(NTHREADS, 2) void k_bwd_walk(KP p, const float* __restrict__ dy_ws, float* __restrict__ dstates,
                                                          float* __restrict__ dm, float* __restrict__ dh0_dir, int walks) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef BwdWalkSmem<PT, BF> SM;
  SM& s = *reinterpret_cast<SM*>(smem_raw);
  constexpr int LDT = SM::LDT, G4 = 4 * PT, ROWS = 4 * PT;
  typedef typename std::conditional<BF, uint16_t, float>::type T;
  typedef typename std::conditional<BF, uint2, f4>::type V;   // four elements of a row
  warm_args();
  if ((int)blockIdx.x >= walks) {
    dm_unit<PT, BF, FULL>(p, dy_ws, dm, (int)blockIdx.x - walks);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cm = lane & 15, g4 = lane >> 4;
  const int nsl = (p.N + NS - 1) / NS;
  // heads fastest: they share C's slice; then the slices, which share the head's dy and x
  unsigned id = xcd_remap(blockIdx.x, walks);
  Unit u;
  u.h = (int)p.by_H(id);
  const int ns = (int)p.by_slices(id);
  u.bt = (int)id;
  u.dir = u.bt & (p.ndir - 1);
  u.b = u.bt >> (p.ndir - 1);
  unsigned g = (unsigned)u.h;
  p.by_hpg(g);
  u.g = (int)g;
  const int n = ns * NS + wave * 16 + cm;
  const bool vn = FULL || n < p.N;
  const Coef cf = lane_coef(p, u.h, n, vn);

  const RowsOf<BF, FULL> ry(p, dy_of(p, u, dy_ws), u);

  // a (P x N) slab of fp32 states; rows past the head dimension read zero and store nothing, as do absent columns
  const unsigned slab = (unsigned)(p.P * p.N) * 4u, nb = (unsigned)p.N * 4u;
  const unsigned at = vn ? (unsigned)(4 * g4 * p.N + n) * 4u : 0x80000000u;
  auto buffer = [](const float* q, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)const_cast<float*>(q), 0, bytes, 0x00027000);
  };
  auto slab_load = [&](const float* q, float (&v)[ROWS]) {
    const __amdgpu_buffer_rsrc_t rs = buffer(q, slab);
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
      v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at + (unsigned)(16 * (k >> 2) + (k & 3)) * nb, 0, 0));
  };
  auto slab_store = [&](float* q, const f4 (&v)[PT]) {
    const __amdgpu_buffer_rsrc_t rs = buffer(q, slab);
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[k >> 2][k & 3]), rs, at + (unsigned)(16 * (k >> 2) + (k & 3)) * nb, 0, 0);
  };

  // what a chunk reads, in the types it is stored in: requested a chunk ahead
  RowMap rm;
  T r_dt[16], r_c[16];
  V r_dy[PT];
  auto request = [&](int c) {
    u.c = c;
    rm = make_rowmap<FULL>(p, u, g4, ns * NS);
    lane_load_raw<BF>(p.dt, u.b, u.h, n, vn, rm, r_dt);
    lane_load_raw<BF>(p.Cm[u.dir], u.b, u.g, n, vn, rm, r_c);
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
      r_dy[i] = ry.get(c, l, p4);
    }
  };

  f4 carry[PT];
  {
    float v[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; ++k) v[k] = 0.0f;
    if (p.dfinal[u.dir]) slab_load(p.dfinal[u.dir] + ((long)u.b * p.H + u.h) * p.P * p.N, v);
#pragma unroll
    for (int k = 0; k < ROWS; ++k) carry[k >> 2][k & 3] = v[k];
  }
  request(p.nc - 1);

  for (int c = p.nc - 1; c >= 0; --c) {
    // ---- dy's tile, transposed
    uint16_t* thi = s.hi[c & 1];
    uint16_t* tlo = s.lo[c & 1];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e4 = tid + i * NTHREADS, l = e4 / G4, p4 = (e4 % G4) * 4;
      const bool ok = ry.has(c, l, p4);
      if constexpr (BF) {
        const uint2 w = ok ? r_dy[i] : make_uint2(0u, 0u);
        thi[p4 * LDT + l] = (uint16_t)w.x;
        thi[(p4 + 1) * LDT + l] = (uint16_t)(w.x >> 16);
        thi[(p4 + 2) * LDT + l] = (uint16_t)w.y;
        thi[(p4 + 3) * LDT + l] = (uint16_t)(w.y >> 16);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float w = ok ? r_dy[i][j] : 0.0f;
          const __bf16 h = (__bf16)w;
          thi[(p4 + j) * LDT + l] = __builtin_bit_cast(uint16_t, h);
          tlo[(p4 + j) * LDT + l] = __builtin_bit_cast(uint16_t, (__bf16)(w - (float)h));
        }
      }
    }
    // ---- dS of the chunk
    slab_store(dstates + dst_off(p, u.bt, c, u.h), carry);
    // ---- the registers the requests went to are free now: the next chunk's leave (at the end chunk 0 once more: in range, unused)
    float raw[16], ct[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      raw[k] = BF ? bf16_to_f((uint16_t)r_dt[k]) : (float)r_dt[k];
      ct[k] = BF ? bf16_to_f((uint16_t)r_c[k]) : (float)r_c[k];
    }
    const RowMap rc = rm;
    request(max(c - 1, 0));
    // ---- C exp(cs) and the chunk's decay
    float total;
    {
      float dtp[16], cs[16], dummy[16];
      total = lane_prep<false>(p, cf, vn, cm, g4, rc, raw, dtp, cs, dummy);
#pragma unroll
      for (int k = 0; k < 16; ++k) ct[k] *= ex2(cs[k]);
    }
    __syncthreads();
    const float e = ex2(total);
#pragma unroll
    for (int pt = 0; pt < PT; ++pt)
#pragma unroll
      for (int r = 0; r < 4; ++r) carry[pt][r] *= e;
    rows_product_split<PT, LDT, BF ? 0 : 1>(carry, thi, tlo, [&](int k) { return ct[k]; }, cm, g4);
  }
  slab_store(dh0_dir + (((long)u.dir * p.B + u.b) * p.H + u.h) * p.P * p.N, carry);
}

bool bwd_walk_available(const KP& p, const float* dy_ws) {
  auto rows_of_four = [](const TensorD& t, int bf) {
    return ((t.s0 | t.s1 | t.s2) & 3) == 0 && ((uintptr_t)t.ptr & (bf ? 7 : 15)) == 0;
  };
  if (p.seq_idx || p.io_dt != p.dt_dt || (p.P & 3) || (dy_ws && p.io_dt)) return false;
  for (int d = 0; d < p.ndir; ++d)
    if (!rows_of_four(p.x[d], p.io_dt) || (!dy_ws && !rows_of_four(p.dout[d], p.io_dt))) return false;
  return true;
}

int launch_bwd_walk(const KP& p, const float* dy_ws, float* dstates, float* dm, float* dh0_dir, hipStream_t st) {
  const int walks = p.B * p.ndir * p.H * ((p.N + NS - 1) / NS), blocks = walks + p.B * p.ndir * p.nc * p.H;
  ISSM_DISPATCH(p, {
    if constexpr (IOB_ == DTB_) {
      constexpr auto kern = &k_bwd_walk<PT_, IOB_, FULL_>;
      hipLaunchKernelGGL(kern, dim3(blocks), dim3(NTHREADS), sizeof(BwdWalkSmem<PT_, IOB_>), st, p, dy_ws, dstates, dm, dh0_dir,
                         walks);
    }
  });
  return (int)hipGetLastError();
}

}  // namespace issm
