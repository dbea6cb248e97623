// Chunk backward of the ISSM scan in tile-base form (gfx950): ddt, dB, dC and the partial sums of dA / ddt_bias.
//
// Same job and same workgroup shape as k_bwd_chunk (issm_bwd.hip): workgroup = (batch, chunk, group, 64 state columns)
// of one direction, looping over the heads of the group; lane (cm, g4) of a wave owns state column cm and the 16 chunk
// rows {16J + 4 g4 + j}.  What differs is how the decay exp2(cs[l] - cs[s]) inside the sums
//   F[l] = sum_{s<=l} dM[l,s] Bd[s] exp2(cs[l]-cs[s]),   G[s] = sum_{l>=s} dM[l,s] C[l] exp2(cs[l]-cs[s])
// is taken apart.  With pc = running sum of a = dt' A log2(e) from the middle of the row's half of the chunk (32 rows; the middle
// of its sum: pc runs from minus half of the half's sum to half of it),
//   exp2(cs[l] - cs[s]) = up[l] . iup[s],  up = exp2(pc), iup = exp2(-pc), for rows of one half, and with
//   across = exp2(half the halves' sums added up) between the two for rows of both.
// up and iup are two exponentials per element, and a row tile's F or G is two chains of plain 16x16x16 products of dM blocks with
// the tiles' operand rows (Bd iup for F, C up for G): the other half's blocks, times across, then those of its own half, all in
// one accumulator -- no per-level operands, no pairs evaluated in the vector ALU.  The state terms fit the same form: exp2(cs[l])
// = up[l] from_start, exp2(cs_last - cs[s]) = to_end iup[s].  (With a reference per tile a block was scaled by its own factor,
// ten exponentials and 20 scaled blocks a head: 5 % more vector instructions, and a wait for every block's result before the next.
// Training steps, 8 x 1024 tokens, 8 heads x 32, 256 states, both directions, fp32 502 -> 496 us; 2 x 16384, bf16, 843 -> 838; heads
// of 36, both directions, bf16, 427 either way; 4 x 1000, 200 states, fp32 203.4 and 203.9.)
//
// up and iup reach 2^(half of the decay across a half), so the form is only used where every 16-row tile's sum stays within
// SPAN_LIMIT (|tt| <= 96, a half's then within twice that: operands below 2^96, no overflow before the factors meet).  A head of a
// workgroup where some column exceeds it -- very large dt' |A| -- is left out here, marked in `redo`, and evaluated by the level-hierarchy kernel
// (k_bwd_chunk / k_bwd_chunk_bf with `redo`), which has no such limit.  Operands, complete tiles: bf16 inputs -> one bf16
// instruction per block, operands rounded once; fp32 inputs -> operands as (hi, lo) bf16 pairs (17 significand
// bits and more), a.b = (ah.bl + al.bh) + (ah.bh + al.bl), each bracket one K = 32 instruction.  Incomplete tiles, four fp32 head
// tiles, and a gated dy: the level form evaluates these calls wherever this kernel cannot, close pairs of rows (bf16 inputs) or all pairs
// (fp32 inputs) from fp32 operands, and what a pair is computed in is not to depend on the kernel.  So the diagonal blocks
// (bf16 inputs) or all blocks (fp32 inputs) are fp32 matrix instructions there.  That costs less than it saves: no operand is
// split, and the 90 - 130 bytes a lane that the pairs of the incomplete form spilled are gone.  d/d(cs) is formed as (operand
// as the matrix instruction took it) x (product) on both rows of a pair, so the two entries of a pair cancel to fp32 rounding
// in the suffix sums.
//
// Built for x / dout rows that allow 8- / 16-byte accesses, x / B / C and dt of one type, no packed sequences, and for bf16
// inputs no z gate; every other call takes the level-hierarchy kernel alone.  That is what lets the kernel issue every
// global load of a head without a branch, one head ahead: the wave then knows how many requests are outstanding at every
// point and waits for exactly the ones it needs (a load inside a branch, even a uniform one, makes the compiler wait for
// all outstanding loads at the join).  Incomplete tiles (FULL = false) run the same code: rows past the end are read through
// a buffer whose bounds check returns zero, columns past the end read column 0 and have dt' = 0, stores are guarded in the
// workgroups that have such rows or columns.  8 x 1024 tokens, 8 heads x 32, one direction: N = 250 104 us fp32, 83 us bf16
// (107 and 86 with operand pairs, 147 and 111 in the level form; N = 256: 88 and 59 us); N = 256 with a gated dy, fp32: 99 us
// (88 with operand pairs, 122 in the level form).
// The lane's own LDS values in 16-byte accesses, rows of x and dy through buffers (their addresses took branches, 64-bit products and, in
// them, waits for the kernel's arguments) and marks that no lane condition holds up: both directions, 8 x 1024 tokens, 8 heads x 32, 256
// states, fp32 172 -> 161 us; heads of 36, bf16 134 -> 131; the training steps of 16 x 2048 tokens, 16 heads x 64, 512 states 8993 -> 8948.
//
// What reaches the chunk's total decay through the states is formed here as well (see `gsum`), from dS, H and the state terms'
// products: the recurrences need not read the states for it (33 - 60 % of their bytes), and what cancels does so exactly: ddt_bias
// and dA of 2 x 512 tokens, 8 heads x 32, 256 states, fp32, 1.7e-4 and 8e-5 -> 6e-6 of their norm from float64; with A a hundred
// times larger 9e-2 and 0.4 -> 2e-4 and 8e-4.
#include <algorithm>

#include "issm_bwd_dx.h"

namespace issm {

constexpr float SPAN_LIMIT = 96.0f;

template <int PT, bool SPLIT>
struct BwdTileSmem {
  static constexpr int KW = 16 * PT, LDP = KW + 8;  // x / dy tiles [l][p]
  // Per-lane values in pieces of four, [k / 4][tid][k % 4]: one 16-byte access each.  In front: an access carries up to 64 KB of its address,
  // and what lies behind costs another register.
  f4 dbc[8 * NTHREADS];      // dB / dC accumulators, k < 16: dB, then dC
  __device__ __forceinline__ float dbc_at(int k, int tid) const { return dbc[(k >> 2) * NTHREADS + tid][k & 3]; }
  // bf16 inputs: the group's B and C values of every lane, packed in pairs (i < 8: B, then C).
  // They are the same for every head of the group; read from global memory again per head they miss the L2 (the heads'
  // streams have been through it in between) and were a third of the kernel's reads; of three and four head tiles, 8 x 1024 tokens,
  // both directions, they cost 76 and 84 us where this takes 71 and 75 (four tiles 84 and 91: 78 and 84; 1000
  // tokens, 250 states, by the kernel trace, three 95 and 102: 85 and 92, four 107 and 118: 99 and 106).
  static constexpr bool BCL = !SPLIT;
  uint4 bc[BCL ? 4 * NTHREADS : 0];
  __device__ __forceinline__ uint2 bc_of(int q, int tid) const { return reinterpret_cast<const uint2*>(bc + (q >> 1) * NTHREADS + tid)[q & 1]; }   // pairs 2 q, 2 q + 1
  // fp32 inputs of up to three head tiles: the B values; C has no room (8 x 1024 tokens, 8 heads x 32, 256 states, both
  // directions, training step 480 -> 466 us, per direction 90 and 100 -> 85 and 94; heads of 48 105 and 112 -> 94 and 104.  It is the
  // 32 registers that B takes neither ahead of a head nor through it, and the loads).
  static constexpr bool BL = SPLIT && PT <= 3;
  f4 bl[BL ? 4 * NTHREADS : 0];
  // T[i][j] = dM[max(i,j)][min(i,j)]; fp32 inputs: hi and lo of four columns side by side, the operand (hi | lo) of a K = 32 instruction as
  // one 16-byte read.  (With the two in matrices of their own every second operand took moves, as the heads a set of zeros for the
  // case that nothing is evaluated: 100 of 1500 vector instructions a head.  8 x 1024 tokens, 8 heads x 48, 256 states, both directions, by
  // direction 105 and 114 -> 101 and 111 us.)
  static constexpr int LDM = CS + (SPLIT ? 4 : 8);
  static constexpr int NH = SPLIT ? 2 : 1;          // hi (and lo) copies
  // fp32 inputs: x and dy one after the other in one place.  (The last rows of the arrays go without
  // padding, and three head tiles then take exactly half of a CU's 160 KB.)
  uint16_t xs[NH * CS * LDP - (SPLIT ? 8 : 0)];
  uint16_t dys_own[SPLIT ? 0 : NH * CS * LDP];
  __device__ __forceinline__ uint16_t* dys() { return SPLIT ? xs : dys_own; }
  alignas(16) uint16_t tm[NH * CS * LDM];
  static constexpr int LDF = CS + 4;                // the same matrix in fp32 (fp32 inputs, incomplete tiles)
  static_assert(!SPLIT || CS * LDF * sizeof(float) <= sizeof(tm), "it takes the pairs' place");
  __device__ __forceinline__ float* tf() { return reinterpret_cast<float*>(tm); }
  int bad[4];                // per wave: some column of the head exceeds SPAN_LIMIT
  int shared[4];             // per wave: some head was left to the level form
};

// Both directions in one workgroup: what a half hands to the other lies behind the two or, without room, in the place of x / dy.
constexpr int DUAL_EX_BYTES = 8 * NTHREADS * sizeof(float);
template <typename SM>
constexpr bool dual_ex_in_tiles() { return 2 * (sizeof(SM) + DUAL_EX_BYTES) > 160 * 1024; }
template <typename SM>
constexpr size_t dual_lds() { return 2 * sizeof(SM) + (dual_ex_in_tiles<SM>() ? 0 : 2 * DUAL_EX_BYTES); }

// An fp32 value rounded to 17 significand bits; a NaN may come out as zero.  (Where it stands below the conversion alone gives
// the same number but for ties; without it the kernel spills 200 bytes a lane instead of 20.)
__device__ __forceinline__ float round17(float v) { return __uint_as_float((__float_as_uint(v) + 0x40u) & 0xffffff80u); }

__device__ __forceinline__ bf8 cat_bf4(bf4 a, bf4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// (v a) b: from one half's scale, up to 2^96, to the other's, down to 2^-96, by two decays whose product may lie below the type's
// range -- where the decay between the rows on either side of the border does not -- and which -ffast-math would form.
__device__ __forceinline__ f4 scaled_twice(f4 v, float a, float b) {
#pragma clang fp reassociate(off)
  f4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float t = v[i] * a;
    r[i] = t * b;
  }
  return r;
}

constexpr int DUAL_TILES = 8, PAIR_TILES = 16;
// PAIR: the workgroups from `blocks` on compute dx (k_bwd_dx_body) of a unit each.  The two do not depend on each other, and where they
// fit the CUs side by side dx costs nothing: kernels of a training step, fp32, 2 x 160 tokens, 4 heads x 32, 128 states 75.7 -> 64.4 us, 2 x 1000,
// 4 x 36, 200 states 115 -> 101; and a launch less to issue.
struct DxPart {
  const float* cabt;
  float* partD;
  int blocks;
};
// PNF: the head dimension fills its 16-row tiles (P == 16 PT); ACC: ddt holds the other direction's share already and
// this launch adds to it; P32 (bf16 only): that share travels in fp32 through p.ddt_part -- the first direction's launch
// writes it there, the second reads it from there and writes the once-rounded sum to ddt.
// TILES: head tiles, DUAL_TILES more (DUAL) for both directions in one launch, four waves each of a workgroup of eight, on the same tokens, head by head: dt comes from memory
// once and their ddt is added up through LDS instead of being stored, read back and stored again (711 -> 510 MB at 8 x 1024 tokens, 8
// heads x 32, 256 states, fp32).  What it gives is less than that, for eight waves now meet where four did: the two launches 88 + 96 us,
// this one 172; heads of 36, bf16, 71 + 75 and 134.  (The second direction a barrier or two behind the first, so that they use LDS and
// the vector ALU at different times: 169, for a barrier then waits for the longer of two different phases.)
// PAIR_TILES more (PAIR): two heads of the group side by side, four waves each of a workgroup of eight, and their sums of dB and dC added up through
// LDS at the end.  For grids that give no CU a second workgroup, where a lone wave a SIMD waits for itself: 2 x 160 tokens, 4 heads x 32, 128
// states, fp32 34.2 -> 24.9 us; 2 x 1000, 4 x 36, 200 states 40.7 -> 31.1; 4 x 1000, 4 x 32, 256 states, bf16 33.1 -> 26.3.
// FULL: complete chunks and column slices; otherwise rows and columns may be absent (see RowMap).  PARTS: gridDim.y workgroups
// share the group's heads, heads_each each (a variant of its own: the two loop bounds more cost the others 25 - 50 scalar
// registers spilled and 1 - 2 % of a training step).
template <int TILES, bool IOB, bool PNF, bool ACC, bool P32, bool FULL, bool PARTS>
__global__ __launch_bounds__(TILES >= DUAL_TILES ? 2 * NTHREADS : NTHREADS, 2) void k_bwd_tile(KP p, const float* __restrict__ states,
                                                          const float* __restrict__ dstates,
                                                          const float* __restrict__ dm, float* __restrict__ partA,
                                                          float* __restrict__ partBias, int* __restrict__ redo, int heads_each, DxPart dx) {
  constexpr bool DUAL = TILES / DUAL_TILES == 1, PAIR = TILES / PAIR_TILES == 1, TWO = DUAL || PAIR;
  static_assert(!PAIR || !PARTS, "one or the other");
  constexpr int PT = TILES % DUAL_TILES;
  if constexpr (PAIR) {
    if ((int)blockIdx.x >= dx.blocks)
      return k_bwd_dx_body<PT, IOB, IOB, FULL, 2>(p, (int)blockIdx.x - dx.blocks, (int)gridDim.x - dx.blocks, nullptr, dstates, dx.cabt, dx.partD);
  }
  const int nblocks = PAIR ? dx.blocks : (int)gridDim.x;
  constexpr bool SPLIT = !IOB;
  // fp32 products in the diagonal blocks / in all blocks.  (Four head tiles, complete: as the level form, which took these calls
  // before, has the closest pairs in fp32.  Operand pairs would leave ddt, dB, dC 5.0 -> 5.4e-6 of their norm from float64, fp32 products
  // 4.9e-6; of 9.55 ms of training step with the level form, 16 x 2048 tokens, 16 heads x 64, 512 states, 9.09 and 9.2 are left.)
  constexpr bool DIAG32 = IOB && !FULL, ALL32 = SPLIT && (!FULL || PT >= 4);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef BwdTileSmem<PT, SPLIT> SM;
  const int half = TWO ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / NTHREADS) : 0;
  SM& s = *reinterpret_cast<SM*>(smem_raw + half * sizeof(SM));
  constexpr int LDP = SM::LDP, LDM = SM::LDM, KT = (PT + 1) / 2;
  constexpr bool BCL = SM::BCL, BL = SM::BL, EX_IN_TILES = dual_ex_in_tiles<SM>();
  static_assert(!EX_IN_TILES || sizeof(s.xs) >= DUAL_EX_BYTES, "it fits");
  // fp32 inputs take turns: x and dS make Q, then dy and H, which are requested at the head's start and not a head
  // ahead, make R in the same place: two barriers a head more.  With all four at once the prefetch spills 76 bytes a lane at three
  // head tiles, each reload waiting for every request before it, and at four the tiles leave one workgroup a CU.  8 x 1024 tokens, 8
  // heads, 256 states, both directions, per direction: heads of 48 128 and 137 -> 104 and 112 us; of 64, which took the level form, 135
  // -> 114 and 121; of 32 the same as before, but it makes room for B (SM::BL).
  constexpr int KP_ = PT * 4;  // dS / H values per lane
  const int tid = TWO ? threadIdx.x % NTHREADS : threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cm = lane & 15, g4 = lane >> 4;
  const int nsl = (p.N + NS - 1) / NS;
  Unit u;
  int wg = xcd_remap(blockIdx.x, nblocks);
  unsigned id = wg;
  const int ns = (int)p.by_slices(id);
  u.g = (int)p.by_G(id);
  u.dir = DUAL ? half : p.dir0;
  u.c = (int)p.by_nc(id);
  u.b = (int)id;
  if (DUAL && half) {   // the same tokens: the mirrored chunk, marked where a launch of this direction alone would
    u.c = p.nc - 1 - u.c;
    wg = ((u.b * p.nc + u.c) * p.G + u.g) * nsl + ns;
  }
  u.bt = u.b * p.ndir + u.dir;
  u.h = u.g * p.hpg;
  const int n = ns * NS + wave * 16 + cm;
  const bool vn = FULL || n < p.N;
  const int nc_ = FULL ? n : (vn ? n : 0);   // where an absent column reads its per-column values
  const RowMap rm = make_rowmap<FULL>(p, u, g4, ns * NS);

#pragma unroll
  for (int q = 0; q < 8; ++q) s.dbc[q * NTHREADS + tid] = (f4){0.0f, 0.0f, 0.0f, 0.0f};

  if (DIAG32) s.shared[wave] = 0;

  if constexpr (BL) {
    float tb[16];
    lane_load_ln<false>(p.Bm[u.dir], u.b, u.g, n, vn, g4, rm, tb);
#pragma unroll
    for (int q = 0; q < 4; ++q) s.bl[q * NTHREADS + tid] = (f4){tb[4 * q], tb[4 * q + 1], tb[4 * q + 2], tb[4 * q + 3]};
  }
  if constexpr (BCL) {
    float tb[16], tc[16];
    lane_load_ln<true>(p.Bm[u.dir], u.b, u.g, n, vn, g4, rm, tb);
    lane_load_ln<true>(p.Cm[u.dir], u.b, u.g, n, vn, g4, rm, tc);
    auto packed = [&](const float (&v)[16], int q) {   // exact: the values are bf16 numbers
      return make_uint4(pack_bf16(v[8 * q], v[8 * q + 1]), pack_bf16(v[8 * q + 2], v[8 * q + 3]), pack_bf16(v[8 * q + 4], v[8 * q + 5]),
                        pack_bf16(v[8 * q + 6], v[8 * q + 7]));
    };
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      s.bc[q * NTHREADS + tid] = packed(tb, q);
      s.bc[(2 + q) * NTHREADS + tid] = packed(tc, q);
    }
  }

  // the reversed direction's launch follows the forward one's and shares dt, x, B, C and ddt with it: it walks the
  // heads backwards, so what the first launch touched last (and the last-level cache still holds) is read first
  auto head_of = [&](int hh) { return u.g * p.hpg + (!DUAL && p.dir0 ? p.hpg - 1 - hh : hh); };

  // Everything a head reads from global memory is requested one head ahead, at the point of the previous head where
  // few registers are live (after its matrix products), so that the requests are in flight while that head's suffix
  // sums and stores run.  (B and C of the lane's rows are the same for every head of the group.  They come out of the workgroup's LDS
  // copy; what has no room there -- C of fp32 inputs, B too for heads of four tiles -- is fetched again per head, from the cache,
  // rather than held in 16 or 32 registers across the loop.)
  // What one head reads: the thread's share of the tiles the four waves stage in LDS (T: rows tid >> 3 and
  // 32 + (tid >> 3), columns 8 (tid & 7) .. + 7 of the hi -- and lo -- matrix; x, dy: group i of the thread is row
  // e4 / 4PT, columns 4 (e4 % 4PT) .. + 3 with e4 = tid + 256 i) and the lane's column operands.  Requested in the order
  // of first use, without a branch; rows of x / dy past the head dimension are read from the tensor's first elements and
  // count as zero.
  uint4 l_th0, l_th1, l_tl0, l_tl1;
  f4 l_xv[SPLIT ? PT : 1], l_dv[SPLIT ? PT : 1];
  uint2 l_nx[SPLIT ? 1 : PT], l_ny[SPLIT ? 1 : PT];
  float l_raw[16], l_A, l_bias, l_dsv[KP_], l_hv[KP_], l_Bv[BCL || BL ? 1 : 16], l_Cv[BCL ? 1 : 16];
  // x and dy: the chunk's rows of a head behind a buffer's base, the first in memory first; pieces that do not exist read zero
  auto rows = [&](const TensorD& t, int h) {
    const int first = u.dir ? p.L - u.c * CS - (FULL ? CS : rm.nvalid) : u.c * CS;
    const char* q = (const char*)t.ptr + ((long)u.b * t.s0 + (long)h * t.s2 + (long)first * t.s1) * (IOB ? 2 : 4);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(q), 0, 0xfffffffcu, 0x00027000);
  };
  auto row_piece = [&](int e4, int s1) -> unsigned {   // four elements, where the thread's group e4 of a tile is
    constexpr int G4 = 4 * PT;
    const int l = e4 / G4, p4 = (e4 % G4) * 4, r = u.dir ? (FULL ? CS : rm.nvalid) - 1 - l : l;
    const bool ok = (PNF || p4 < p.P) && (FULL || l < rm.nvalid);
    return ok ? (unsigned)(r * s1 + p4) * (IOB ? 2u : 4u) : 0xfffffffcu;
  };
  auto request_dy_h = [&](int h) {   // fp32 inputs: the operands of R
    int tq = tid;
    asm volatile("" : "+v"(tq));
    const __amdgpu_buffer_rsrc_t rs = rows(p.dout[u.dir], h);
    const int sy = (int)p.dout[u.dir].s1;
#pragma unroll
    for (int i = 0; i < PT; ++i)
      l_dv[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, row_piece(tq + i * NTHREADS, sy), 0, 0));
    lane_load_pn<KP_>(states + st_off(p, u.bt, u.c, h), p.P, p.N, n, vn, g4, PNF, l_hv);
  };
  auto request = [&](int hnext) {
    int tq = tid;
    asm volatile("" : "+v"(tq));
    const char* dmb = reinterpret_cast<const char*>(dm + sq_off(p, u.bt, u.c, hnext));
    const unsigned mo = (unsigned)tq * 16u;
    l_th0 = *(const uint4*)(dmb + mo);
    l_th1 = *(const uint4*)(dmb + (mo + 32u * CS * 2u));
    if constexpr (SPLIT) {
      l_tl0 = *(const uint4*)(dmb + (mo + CS * CS * 2u));
      l_tl1 = *(const uint4*)(dmb + (mo + (CS * CS + 32u * CS) * 2u));
    }
    {
      const __amdgpu_buffer_rsrc_t rx = rows(p.x[u.dir], hnext);
      const int sx = (int)p.x[u.dir].s1;
      if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < PT; ++i)
          l_xv[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rx, row_piece(tq + i * NTHREADS, sx), 0, 0));
      } else {
        const __amdgpu_buffer_rsrc_t ry = rows(p.dout[u.dir], hnext);
        const int sy = (int)p.dout[u.dir].s1;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          l_ny[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(ry, row_piece(tq + i * NTHREADS, sy), 0, 0));
          l_nx[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rx, row_piece(tq + i * NTHREADS, sx), 0, 0));
        }
      }
    }
    lane_load_ln<IOB>(p.dt, u.b, hnext, n, vn, g4, rm, l_raw);
    l_A = p.A[hnext * p.N + nc_];
    {
      const float* bp = p.dt_bias ? p.dt_bias : p.A;  // no bias: any readable address, the value is dropped
      const float b = bp[hnext * p.N + nc_];
      l_bias = p.dt_bias ? b : 0.0f;
    }
    lane_load_pn<KP_>(dstates + dst_off(p, u.bt, u.c, hnext), p.P, p.N, n, vn, g4, PNF, l_dsv);
    if constexpr (!SPLIT) lane_load_pn<KP_>(states + st_off(p, u.bt, u.c, hnext), p.P, p.N, n, vn, g4, PNF, l_hv);
    if constexpr (!BCL) {
      if constexpr (!BL) lane_load_ln<IOB>(p.Bm[u.dir], u.b, u.g, n, vn, g4, rm, l_Bv);
      lane_load_ln<IOB>(p.Cm[u.dir], u.b, u.g, n, vn, g4, rm, l_Cv);
    }
  };
  // the thread's share of a (64 x 16 PT) tile as (hi, lo) pairs into LDS
  auto put_split = [&](const f4 (&v)[SPLIT ? PT : 1], uint16_t* dst, int tq) {
    if constexpr (SPLIT) {
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int e4 = tq + i * NTHREADS, o = (e4 / (4 * PT)) * LDP + (e4 % (4 * PT)) * 4;
        const float w[4] = {v[i][0], v[i][1], v[i][2], v[i][3]};
        bf4 h, l;
        split4(w, h, l);
        *(bf4*)(dst + o) = h;
        *(bf4*)(dst + CS * LDP + o) = l;
      }
    }
  };
  // (PAIR: heads_each is half of an even number, so that both halves of the workgroup meet at the same barriers)
  const int hh0 = PARTS ? (int)blockIdx.y * heads_each : PAIR ? half * heads_each : 0;
  request(head_of(hh0));

  for (int hh = hh0; hh < (PARTS ? min(p.hpg, hh0 + heads_each) : PAIR ? hh0 + heads_each : p.hpg); ++hh) {
    u.h = head_of(hh);
    __syncthreads();  // the previous head no longer reads the tiles
    {
      int tq = tid;
      asm volatile("" : "+v"(tq));
      const int mrow = tq >> 3, mcol = (tq & 7) * 8;
      constexpr int G4 = 4 * PT;
      if constexpr (ALL32) {  // T = hi + lo as fp32 numbers
        auto put = [&](int row, uint4 h, uint4 l) {
          const unsigned a[4] = {h.x, h.y, h.z, h.w}, b[4] = {l.x, l.y, l.z, l.w};
          f4 v[2];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i >> 1][(2 * i) & 3] = __uint_as_float(a[i] << 16) + __uint_as_float(b[i] << 16);
            v[i >> 1][(2 * i + 1) & 3] = __uint_as_float(a[i] & 0xffff0000u) + __uint_as_float(b[i] & 0xffff0000u);
          }
          f4* d = (f4*)(s.tf() + row * SM::LDF + mcol);
          d[0] = v[0];
          d[1] = v[1];
        };
        put(mrow, l_th0, l_tl0);
        put(32 + mrow, l_th1, l_tl1);
      } else {
        if constexpr (SPLIT) {
          uint2* d0 = (uint2*)(s.tm + 2 * (mrow * LDM + mcol));
          uint2* d1 = (uint2*)(s.tm + 2 * ((32 + mrow) * LDM + mcol));
          d0[0] = make_uint2(l_th0.x, l_th0.y); d0[1] = make_uint2(l_tl0.x, l_tl0.y);
          d0[2] = make_uint2(l_th0.z, l_th0.w); d0[3] = make_uint2(l_tl0.z, l_tl0.w);
          d1[0] = make_uint2(l_th1.x, l_th1.y); d1[1] = make_uint2(l_tl1.x, l_tl1.y);
          d1[2] = make_uint2(l_th1.z, l_th1.w); d1[3] = make_uint2(l_tl1.z, l_tl1.w);
        } else {
          *(uint4*)(s.tm + mrow * LDM + mcol) = l_th0;
          *(uint4*)(s.tm + (32 + mrow) * LDM + mcol) = l_th1;
        }
      }
      if constexpr (SPLIT) {
        put_split(l_xv, s.xs, tq);
      } else {
        lp_store_raw<PT, LDP>(l_ny, s.dys(), tq);
        lp_store_raw<PT, LDP>(l_nx, s.xs, tq);
      }
    }
    if constexpr (SPLIT) request_dy_h(u.h);

    // ---- dt transform and the per-tile running sums, before the barrier that publishes the tiles: the same barrier
    // then also publishes whether any column of the workgroup is out of the form's range
    Coef cf;
    cf.A = l_A;
    cf.bias = l_bias;
    const float An = cf.A;
    float dtp[16], dfac[16], pc[16], tt[4];
    lane_dt<true>(p, cf, vn, g4, rm, l_raw, dtp, dfac);
    float half0, half1;
    lane_half_sums<IOB>(An * LOG2E, cm, g4, dtp, pc, tt, half0, half1);
    {
      const float worst = fmaxf(fmaxf(fabsf(tt[0]), fabsf(tt[1])), fmaxf(fabsf(tt[2]), fabsf(tt[3])));
      const bool bad = !(worst <= SPAN_LIMIT);  // also true for NaN
      int wq = wave;
      asm volatile("" : "+v"(wq));   // (an address formed here, not kept)
      s.bad[wq] = __any(bad) ? 1 : 0;
    }
    __syncthreads();
    const int4 bd = *(const int4*)s.bad;
    int any_bad = bd.x | bd.y | bd.z | bd.w;
    if constexpr (DUAL) {
      const int4 be = *(const int4*)reinterpret_cast<SM*>(smem_raw + (1 - half) * sizeof(SM))->bad;
      any_bad |= be.x | be.y | be.z | be.w;
    }
    const bool skip = any_bad != 0;  // uniform: the whole head is left to the level-hierarchy kernel
    // (all threads store the one value: a store under a lane condition has the waits for the requests before it wait for the store as well)
    redo[(u.dir * nblocks + wg) * p.hpg + (DUAL && half ? p.hpg - 1 - hh : hh)] = skip ? 1 : 0;
    if (DIAG32 && skip) s.shared[wave] = 1;
    const uint16_t* xs_ = s.xs;
    const uint16_t* dys_ = s.dys();
    const uint16_t* tm_ = s.tm;

    float dcs[16], val[16], gsum = 0.0f;   // gsum: the lane's share of the states' gradient to the chunk's total, see below
    if (skip) {
#pragma unroll
      for (int k = 0; k < 16; ++k) asm volatile("v_mov_b32 %0, 0\nv_mov_b32 %1, 0" : "=v"(dcs[k]), "=v"(val[k]));  // (opaque: zeros set in advance are set for every head)
      if constexpr (PAIR && SPLIT) {   // the other half's head may stand at these
        __syncthreads();
        __syncthreads();
      }
    } else {
      // dS and H of the lane's column as (hi, lo) bf16 pairs: the B operands of Q = x . dS and R = dy . H (products over
      // the head dimension, K = 32 per step; k-slot s of step t <-> lane value 8 t + s).  They are fp32 states, whose rounding to
      // 8 bits would be far above that of the inputs.
      auto state_pairs = [&](const float (&v)[KP_], bf8 (&hi)[KT], bf8 (&lo)[KT]) {
#pragma unroll
        for (int t = 0; t < KT; ++t) {
          float a[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) a[j] = 8 * t + j < KP_ ? v[(8 * t + j) % KP_] : 0.0f;
          split8(a, hi[t], lo[t]);
        }
      };
      f4 qs[SPLIT ? 4 : 1], rs[SPLIT ? 4 : 1];
      if constexpr (SPLIT) {
        int cq = cm, gq = g4, tq = tid;
        asm volatile("" : "+v"(cq), "+v"(gq), "+v"(tq));
        auto rows_times = [&](const bf8 (&hi)[KT], const bf8 (&lo)[KT], f4 (&out)[SPLIT ? 4 : 1]) {
#pragma unroll
          for (int R = 0; R < 4; ++R) {
            f4 q = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < KT; ++t) {
              const bool half = (PT & 1) && t == KT - 1;
              const uint16_t* lo_tile = xs_ + CS * LDP;
              const bf8 xh = half ? split_frag<LDP, true>(xs_, R * 16 + cq, gq, t) : split_frag<LDP>(xs_, R * 16 + cq, gq, t);
              const bf8 xl = half ? split_frag<LDP, true>(lo_tile, R * 16 + cq, gq, t) : split_frag<LDP>(lo_tile, R * 16 + cq, gq, t);
              q = mfma_bf(xh, lo[t], q);
              q = mfma_bf(xl, hi[t], q);
              q = mfma_bf(xh, hi[t], q);
            }
            out[R] = q;
          }
        };
        bf8 hi[KT], lo[KT];
        state_pairs(l_dsv, hi, lo);
        rows_times(hi, lo, qs);
        __syncthreads();   // (skip is the workgroup's or, PAIR, its half's)
        put_split(l_dv, s.dys(), tq);
        gsum = lane_dot_pn<KP_>(l_dsv, l_hv, p.P, g4, PNF);
        state_pairs(l_hv, hi, lo);
        __syncthreads();
        rows_times(hi, lo, rs);
      }
      // ---- decay factors and the operand rows
      __builtin_amdgcn_sched_barrier(0);
      float up[16], iup[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        up[k] = ex2(pc[k]);
        iup[k] = ex2(-pc[k]);
      }
      // decays of half a half; from a half's middle to its end, or from its start to its middle
      const float e0 = ex2(half0), e1 = ex2(half1);
      const float across = e0 * e1;                        // from the middle of the first half to that of the second
      const float from_start[2] = {e0, e0 * across};       // from the chunk's start to the middles
      const float to_end[2] = {across * e1, e1};           // from the middles to the chunk's end
      auto unpk = [](const unsigned (&a)[8], int k) {
        return __uint_as_float((k & 1) ? (a[k >> 1] & 0xffff0000u) : (a[k >> 1] << 16));
      };
      auto wide = [](uint2 a) -> f4 {  // four bf16 numbers
        return (f4){__uint_as_float(a.x << 16), __uint_as_float(a.x & 0xffff0000u), __uint_as_float(a.y << 16),
                    __uint_as_float(a.y & 0xffff0000u)};
      };
      auto b_tile = [&](int R) {   // B of the lane's rows of tile R
        if constexpr (BL) return s.bl[R * NTHREADS + tid];
        else return (f4){l_Bv[BCL ? 0 : 4 * R], l_Bv[BCL ? 0 : 4 * R + 1], l_Bv[BCL ? 0 : 4 * R + 2], l_Bv[BCL ? 0 : 4 * R + 3]};
      };
      // Cu = C up (operand of the G blocks), Bi = B dt' iup (operand of the F blocks)
      bf4 Ch[4], Bh[4], Cl[4], Bl[4];
      float cf32[ALL32 ? 16 : 1], bf32[ALL32 ? 16 : 1];
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        f4 b4, c4;
        if constexpr (!BCL) {
          b4 = b_tile(J);
          c4 = (f4){l_Cv[4 * J], l_Cv[4 * J + 1], l_Cv[4 * J + 2], l_Cv[4 * J + 3]};
        } else {  // out of the workgroup's LDS copy of the group's B and C
          b4 = wide(s.bc_of(J, tid));
          c4 = wide(s.bc_of(4 + J, tid));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = 4 * J + j;
          const float cu = c4[j] * up[k], bi = b4[j] * dtp[k] * iup[k];
          if constexpr (ALL32) {
            cf32[k] = cu;
            bf32[k] = bi;
            continue;
          }
          Ch[J][j] = (__bf16)(SPLIT ? round17(cu) : cu);
          Bh[J][j] = (__bf16)(SPLIT ? round17(bi) : bi);
          if (SPLIT) {  // of the value itself, rounded to 8 bits: the pair holds it to 2^-18, and what is no number stays none
            Cl[J][j] = (__bf16)(cu - (float)Ch[J][j]);
            Bl[J][j] = (__bf16)(bi - (float)Bh[J][j]);
          }
        }
      }
      // B (and, for bf16 inputs, C) as the column phase needs them: bf16 inputs are bf16 numbers and stay packed, two
      // to a register
      unsigned bvp[8], cvp[8];
      float bvf[SPLIT && !BL ? 16 : 1];
      if constexpr (BCL && DIAG32) {  // read tile by tile below
      } else if constexpr (BCL) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint2 b2 = s.bc_of(q, tid), c2 = s.bc_of(4 + q, tid);
          bvp[2 * q] = b2.x; bvp[2 * q + 1] = b2.y;
          cvp[2 * q] = c2.x; cvp[2 * q + 1] = c2.y;
        }
      } else {
#pragma unroll
        for (int k = 0; k < (BL ? 0 : 16); ++k) bvf[k] = l_Bv[k];
      }
      __builtin_amdgcn_sched_barrier(0);

      int cq = cm, gq = g4;
      asm volatile("" : "+v"(cq), "+v"(gq));
      // The chunk's total decay acts on the states alone, with the gradient sum_p dS H_next = exp2(total) sum_p dS H +
      // sum_l (Bd exp2(total - cs))[l] Q[l]: the second sum is the state terms of the column phase, which cancel against it
      // exactly in the suffix sums, so the next chunk's H is not read and nothing has to be summed over p elsewhere.
      if constexpr (!SPLIT) gsum = lane_dot_pn<KP_>(l_dsv, l_hv, p.P, g4, PNF);
      gsum *= across * across;
      if constexpr (SPLIT) asm volatile("" : "+v"(gsum));   // (8 - 20 bytes a lane of scratch less; bf16 inputs: more)
      bf8 dsh[KT], dsl[KT], hh_[KT], hl_[KT];
      if constexpr (!SPLIT) {
        state_pairs(l_dsv, dsh, dsl);
        state_pairs(l_hv, hh_, hl_);
      }
      unsigned mf[2], mg[2];  // bf16-pair masks of the diagonal block for this lane's four columns 4 g4 + j
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const int c0 = 4 * gq + 2 * w;
        mf[w] = (c0 <= cq ? 0xffffu : 0u) | (c0 + 1 <= cq ? 0xffff0000u : 0u);
        mg[w] = (c0 >= cq ? 0xffffu : 0u) | (c0 + 1 >= cq ? 0xffff0000u : 0u);
      }
      auto block = [&](uint2 ah, uint2 al, bf4 bh, bf4 bl, f4 acc) -> f4 {
        const bf4 a_h = __builtin_bit_cast(bf4, ah);
        if constexpr (SPLIT) {
          // (ah + al) . (bh + bl) in full: the same A fragment against (bl | bh) and (bh | bl).  All four terms, so
          // that F and G see one and the same product dM . B . C (as the instructions took them) for a pair of rows
          const bf8 a2 = cat_bf4(a_h, __builtin_bit_cast(bf4, al));
          acc = mfma_bf(a2, cat_bf4(bl, bh), acc);
          return mfma_bf(a2, cat_bf4(bh, bl), acc);
        } else {
          return mfma_bf16k(a_h, bh, acc);
        }
      };
      // the blocks of two tiles
      auto block2 = [&](const uint2 (&ah)[4], const uint2 (&al)[4], const bf4 (&bh)[4], const bf4 (&bl)[4], int c, f4 acc) -> f4 {
        return block(ah[c + 1], al[c + 1], bh[c + 1], bl[c + 1], block(ah[c], al[c], bh[c], bl[c], acc));
      };

      auto block32 = [&](f4 a, const float* op, f4 acc) -> f4 {  // fp32: k-slot g4 of instruction j <-> row / column 4 g4 + j
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = mfma4(a[j], op[j], acc);
        return acc;
      };
      // the diagonal block's entries on or before (F) / on or after (G) the diagonal, for the lane's columns 4 g4 + j
      auto upto = [&](f4 a) -> f4 {
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = 4 * gq + j <= cq ? a[j] : 0.0f;
        return a;
      };
      auto from = [&](f4 a) -> f4 {
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = 4 * gq + j >= cq ? a[j] : 0.0f;
        return a;
      };

      // ---- tile by tile: the state terms of the lane's four rows of tile R, the blocks of F and G that end in them,
      // and their share of the column phase.  Row block R of T (rows 16 R + cm) serves the F blocks (R, c <= R) and, T
      // being symmetric, the G blocks (c >= R, R); on the diagonal block F keeps the columns <= the row and G those >= it.
#pragma unroll
      for (int R = 0; R < 4; ++R) {
        f4 xf = {0, 0, 0, 0}, xg = {0, 0, 0, 0};  // the blocks' sums
        f4 df = {0, 0, 0, 0}, dg = {0, 0, 0, 0};  // DIAG32: those of the diagonal block
        float cd[4], bd[4];                       // DIAG32: the operands of rows 16 R + 4 g4 + j
        if constexpr (DIAG32) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const uint2 b2 = s.bc_of(R, tid), c2 = s.bc_of(4 + R, tid);
            bvp[2 * R + j] = j ? b2.y : b2.x;
            cvp[2 * R + j] = j ? c2.y : c2.x;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int k = 4 * R + j;
            cd[j] = unpk(cvp, k) * up[k];
            bd[j] = unpk(bvp, k) * dtp[k] * iup[k];
          }
        }
        f4 sf, sg;                                // the state terms
        {
          f4 q = {0, 0, 0, 0}, r = {0, 0, 0, 0};
          if constexpr (SPLIT) {
            q = qs[R];
            r = rs[R];
          }
#pragma unroll
          for (int t = 0; t < (SPLIT ? 0 : KT); ++t) {
            const bool half = (PT & 1) && t == KT - 1;
            const bf8 xfr = half ? split_frag<LDP, true>(xs_, R * 16 + cq, gq, t) : split_frag<LDP>(xs_, R * 16 + cq, gq, t);
            const bf8 yfr = half ? split_frag<LDP, true>(dys_, R * 16 + cq, gq, t) : split_frag<LDP>(dys_, R * 16 + cq, gq, t);
            q = mfma_bf(xfr, dsl[t], q);
            r = mfma_bf(yfr, hl_[t], r);
            q = mfma_bf(xfr, dsh[t], q);
            r = mfma_bf(yfr, hh_[t], r);
          }
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            sg[rr] = to_end[R >> 1] * q[rr];
            sf[rr] = from_start[R >> 1] * r[rr];
          }
        }
        if constexpr (ALL32) {
          const float* row = s.tf() + (16 * R + cq) * SM::LDF + 4 * gq;
          f4 t[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) t[c] = *(const f4*)(row + 16 * c);
          // (as below)
          if (R >= 2) xf = scaled_twice(block32(t[1], bf32 + 4, block32(t[0], bf32, xf)), e0, e1);
          if (R < 2) xg = scaled_twice(block32(t[3], cf32 + 12, block32(t[2], cf32 + 8, xg)), e1, e0);
          const int O = R ^ 1;
          if (R & 1) xf = block32(t[O], bf32 + 4 * O, xf);
          else xg = block32(t[O], cf32 + 4 * O, xg);
          xf = block32(upto(t[R]), bf32 + 4 * R, xf);
          xg = block32(from(t[R]), cf32 + 4 * R, xg);
        } else {
          uint2 th[4], tl[4];
          const uint16_t* row = tm_ + (SPLIT ? 2 : 1) * ((16 * R + cq) * LDM + 4 * gq);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if constexpr (SPLIT) {
              const uint4 t = *(const uint4*)(row + 32 * c);
              th[c] = make_uint2(t.x, t.y);
              tl[c] = make_uint2(t.z, t.w);
            } else {
              th[c] = *(const uint2*)(row + 16 * c);
              tl[c] = make_uint2(0u, 0u);
            }
          }
          // the other half's blocks first: their sum decays across the middles; then those of the rows' own half
          if (R >= 2) xf = scaled_twice(block2(th, tl, Bh, Bl, 0, xf), e0, e1);
          if (R < 2) xg = scaled_twice(block2(th, tl, Ch, Cl, 2, xg), e1, e0);
          const int O = R ^ 1;   // the half's other tile
          const uint2 dh = th[R], dl = tl[R];
          if constexpr (DIAG32) {
            if (R & 1) xf = block(th[O], tl[O], Bh[O], Bl[O], xf);
            else xg = block(th[O], tl[O], Ch[O], Cl[O], xg);
            df = block32(upto(wide(dh)), bd, df);
            dg = block32(from(wide(dh)), cd, dg);
          } else {
            th[R] = make_uint2(dh.x & mf[0], dh.y & mf[1]);
            tl[R] = make_uint2(dl.x & mf[0], dl.y & mf[1]);
            xf = (R & 1) ? block2(th, tl, Bh, Bl, R & 2, xf) : block(th[R], tl[R], Bh[R], Bl[R], xf);
            th[R] = make_uint2(dh.x & mg[0], dh.y & mg[1]);
            tl[R] = make_uint2(dl.x & mg[0], dl.y & mg[1]);
            xg = (R & 1) ? block(th[R], tl[R], Ch[R], Cl[R], xg) : block2(th, tl, Ch, Cl, R & 2, xg);
          }
        }
        // The rows' share of the column phase.  d/d(cs) = C X2 - Bd E1 takes the blocks' sums times the operands as the
        // matrix instructions took them: a pair of rows then enters both of its rows as one and the same product and
        // cancels in the suffix sums to fp32 rounding.  The state terms take, with bf16 inputs, the unrounded operands (B and
        // C are exact, the decays fp32); with fp32 inputs the operand pairs are as accurate as the split products Q and R.
        if constexpr (!SPLIT) __builtin_amdgcn_sched_barrier(0);   // (asked for any earlier, the sums cost 8 to 20 bytes a lane of scratch)
        f4 db4 = s.dbc[R * NTHREADS + tid], dc4 = s.dbc[(4 + R) * NTHREADS + tid], b4;
        if constexpr (BL) b4 = b_tile(R);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int k = 4 * R + rr;
          const float bv = SPLIT ? (BL ? b4[rr] : bvf[SPLIT && !BL ? k : 0]) : unpk(bvp, k);
          const float E1 = iup[k] * (sg[rr] + xg[rr] + dg[rr]), X2 = up[k] * (sf[rr] + xf[rr] + df[rr]);
          db4[rr] += dtp[k] * E1;
          dc4[rr] += X2;
          val[k] = bv * E1;
          if constexpr (ALL32) {
            dcs[k] = cf32[k] * (xf[rr] + sf[rr]) - bf32[k] * (xg[rr] + sg[rr]);
            gsum += bf32[k] * sg[rr];
          } else if constexpr (SPLIT) {
            const float c16 = (float)Ch[R][rr] + (float)Cl[R][rr], b16 = (float)Bh[R][rr] + (float)Bl[R][rr];
            dcs[k] = c16 * (xf[rr] + sf[rr]) - b16 * (xg[rr] + sg[rr]);
            gsum += b16 * sg[rr];
          } else {
            const float c16 = (float)Ch[R][rr], b16 = (float)Bh[R][rr];
            float pairs = c16 * xf[rr] - b16 * xg[rr];
            if constexpr (DIAG32) pairs += cd[rr] * df[rr] - bd[rr] * dg[rr];
            const float own = bv * dtp[k] * iup[k] * sg[rr];
            dcs[k] = pairs + (unpk(cvp, k) * up[k] * sf[rr] - own);
            gsum += own;
          }
        }
        s.dbc[R * NTHREADS + tid] = db4;
        s.dbc[(4 + R) * NTHREADS + tid] = dc4;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    pin16(dcs); pin16(val);

    // ---- this direction's predecessor in ddt, then the next head's requests: all of them stay in flight through the
    // rest of this head, which only waits for the predecessor's values (requested before them)
    float old[16];
    if constexpr (ACC) {
      if constexpr (P32) lane_load_ln<false>(p.ddt_part, u.b, u.h, n, vn, g4, rm, old);
      else lane_load_ln<IOB>(p.ddt, u.b, u.h, n, vn, g4, rm, old);
    }
    request(head_of(min(hh + 1, (PARTS ? min(p.hpg, hh0 + heads_each) : PAIR ? hh0 + heads_each : p.hpg) - 1)));  // (unconditional: the last head is requested again and not used)
    __builtin_amdgcn_sched_barrier(0);
    // DUAL: the two halves of the workgroup have one column's rows in opposite order (row k of a lane of the one is row 15 - k of
    // lane ^ 48 of the other); each hands its first eight over and stores the sums of its last eight.
    auto store_late = [&](const float (&v)[16]) {
      typedef typename std::conditional<IOB, uint16_t, float>::type T;
      T* q = (T*)const_cast<void*>(p.ddt.ptr) + ((long)u.b * p.ddt.s0 + (long)u.h * p.ddt.s2);
      const unsigned lo = (unsigned)(rm.base * (int)p.ddt.s1 + n) * (unsigned)sizeof(T);
      unsigned ks = (unsigned)(rm.step * (int)p.ddt.s1) * (unsigned)sizeof(T);
      ISSM_OPAQUE_S(ks);
#pragma unroll
      for (int k = 8; k < 16; ++k) {
        T* d = (T*)((char*)q + (lo + (unsigned)(16 * (k >> 2) + (k & 3)) * ks));
        if (IOB) *d = (T)f_to_bf16(v[k]); else *d = (T)v[k];
      }
    };
    if (skip) {
      if constexpr (DUAL) {
        store_late(val);
        continue;
      }
      // the level-hierarchy kernel adds this head's share to ddt later: it must find the other direction's, or zero
      if constexpr (!ACC) {  // (val is all zero here)
        if constexpr (P32) lane_store_ln<false>(p.ddt_part, u.b, u.h, n, vn, g4, rm, val);
        else lane_store_ln<IOB>(p.ddt, u.b, u.h, n, vn, g4, rm, val);
      } else if constexpr (P32) {
        lane_store_ln<IOB>(p.ddt, u.b, u.h, n, vn, g4, rm, old);  // the other direction's share moves into ddt
      }
      continue;
    }

    // ---- the rest of the column phase: suffix sums over the rows, ddt, the partial sums
    // (fresh opaque lane coordinates: the cross-lane fetch addresses are formed here rather than kept across the loop and
    // reloaded from scratch behind the requests in flight)
    int cm2 = cm, g42 = g4;
    asm volatile("" : "+v"(cm2), "+v"(g42));
    {
      // suffix sums up the 64 rows, from the gradient to the chunk's total on
      float c[4], v[4], t[4], carry;   // carry: sum over all rows after the current tile
#pragma unroll
      for (int J = 3; J >= 0; --J) {
        float a = 0.0f;
#pragma unroll
        for (int j = 3; j >= 0; --j) {
          a += dcs[4 * J + j];
          dcs[4 * J + j] = a;
        }
        c[J] = a;
      }
      if constexpr (IOB) {
#pragma unroll
        for (int J = 0; J < 4; ++J) t[J] = __shfl_down(c[J], 16, 64);
        gsum += __shfl_xor(gsum, 16, 64);
#pragma unroll
        for (int J = 0; J < 4; ++J) v[J] = g42 <= 2 ? c[J] + t[J] : c[J];
#pragma unroll
        for (int J = 0; J < 4; ++J) t[J] = __shfl_down(v[J], 32, 64);
#pragma unroll
        for (int J = 0; J < 4; ++J) v[J] = g42 <= 1 ? v[J] + t[J] : v[J];  // inclusive from the last lane group down
#pragma unroll
        for (int J = 0; J < 4; ++J) t[J] = __shfl(v[J], cm2, 64);           // tile totals
        carry = gsum + __shfl_xor(gsum, 32, 64);
      } else {
#pragma unroll
        for (int J = 0; J < 4; ++J) {
          float before;
          group_sums(c[J], g42, before, v[J], t[J]);   // of the rows behind, of the tile
        }
        float before, after;
        group_sums(gsum, g42, before, after, carry);
      }
#pragma unroll
      for (int J = 3; J >= 0; --J) {
        const float add = carry + (IOB ? v[J] - c[J] : v[J]);
#pragma unroll
        for (int j = 0; j < 4; ++j) dcs[4 * J + j] += add;
        carry += t[J];
      }
    }
    float sumA = 0.0f, sumB = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float da = dcs[k];
      sumA += da * dtp[k];
      val[k] = (val[k] + da * An) * dfac[k];
      sumB += val[k];
    }
    if constexpr (ACC) {
#pragma unroll
      for (int k = 0; k < 16; ++k) val[k] += old[k];
    }
    if constexpr (DUAL) {
      if constexpr (EX_IN_TILES) __syncthreads();
      f4* ex = reinterpret_cast<f4*>(EX_IN_TILES ? (unsigned char*)s.xs : smem_raw + 2 * sizeof(SM) + half * DUAL_EX_BYTES);
      const f4* ey = reinterpret_cast<const f4*>(EX_IN_TILES ? (const unsigned char*)reinterpret_cast<SM*>(smem_raw + (1 - half) * sizeof(SM))->xs
                                                                       : smem_raw + 2 * sizeof(SM) + (1 - half) * DUAL_EX_BYTES);
      int tq = tid;
      asm volatile("" : "+v"(tq));
#pragma unroll
      for (int q = 0; q < 2; ++q) ex[q * NTHREADS + tq] = (f4){val[4 * q], val[4 * q + 1], val[4 * q + 2], val[4 * q + 3]};
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f4 v = ey[q * NTHREADS + (tq ^ 48)];
#pragma unroll
        for (int j = 0; j < 4; ++j) val[15 - 4 * q - j] += v[j];
      }
      store_late(val);
    } else if constexpr (!ACC && P32) lane_store_ln<false>(p.ddt_part, u.b, u.h, n, vn, g4, rm, val);
    else lane_store_ln<IOB>(p.ddt, u.b, u.h, n, vn, g4, rm, val);
    sumA = scan_g_incl(sumA, g4);
    sumB = scan_g_incl(sumB, g4);
    if (g4 == 3 && vn) {
      // (an opaque copy of the column: the two per-lane addresses are then formed here instead of being kept, as 64-bit
      // values, across the head loop -- a reload from scratch at this point would wait for every request in flight)
      int nq = n;
      asm volatile("" : "+v"(nq));
      partA[vec_off(p, u.bt, u.c, u.h) + nq] = sumA;
      partBias[vec_off(p, u.bt, u.c, u.h) + nq] = sumB;
    }
  }

  if constexpr (PAIR) {   // each half adds up one of the two sums, and stores it
    __syncthreads();
    const SM &s0 = *reinterpret_cast<const SM*>(smem_raw), &s1 = *reinterpret_cast<const SM*>(smem_raw + sizeof(SM));
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = s0.dbc_at(16 * half + k, tid) + s1.dbc_at(16 * half + k, tid);
    if (DIAG32 && p.dbc_part && (s0.shared[wave] | s1.shared[wave])) {
      float* q = p.dbc_part + (long)wg * (32 * NTHREADS) + 16 * half * NTHREADS + tid;
#pragma unroll
      for (int k = 0; k < 16; ++k) q[k * NTHREADS] = v[k];
    } else {
      const TensorD& d = half ? p.dC[u.dir] : p.dB[u.dir];
      if (d.ptr) lane_store_ln<IOB>(d, u.b, u.g, n, vn, g4, rm, v);
    }
    return;
  }
  if (PARTS || (DIAG32 && p.dbc_part && s.shared[wave])) {  // (the wave's own word)
    const long at = (long)p.dir0 * gridDim.x + wg;
    float* q = p.dbc_part + (PARTS ? (long)blockIdx.y * p.ndir * gridDim.x + at : at) * (32 * NTHREADS) + tid;
#pragma unroll
    for (int k = 0; k < 32; ++k) q[k * NTHREADS] = s.dbc_at(k, tid);
  } else {
    float vb[16], vc[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      vb[k] = s.dbc_at(k, tid);
      vc[k] = s.dbc_at(16 + k, tid);
    }
    if (p.dB[u.dir].ptr) lane_store_ln<IOB>(p.dB[u.dir], u.b, u.g, n, vn, g4, rm, vb);
    if (p.dC[u.dir].ptr) lane_store_ln<IOB>(p.dC[u.dir], u.b, u.g, n, vn, g4, rm, vc);
  }
}

// Whether the tile-base kernel is built for this call (otherwise the level-hierarchy kernel does all the work): no packed
// sequences (their cuts are outside the form's range), x / B / C and dt of one type, x and dout rows that allow vector
// accesses, ddt wanted, a gated dy (which is fp32) only beside fp32 inputs.  Four fp32 head tiles, one head a group and one
// direction: the level form, which also has the closest pairs in fp32, is no slower without the pass over the marks (1 x 512
// tokens, 1 head of 64, 256 states 14.9 us against 13.1 + 3.8; 8 x 1024, 2 groups 48.3 against 42.2 + 5.2) and a launch less.
bool bwd_tile_available(const KP& p, const float* dy_ws) {
  if (p.seq_idx || (dy_ws && p.io_dt) || p.io_dt != p.dt_dt || !p.ddt.ptr) return false;
  if (!p.io_dt && p.P > 48 && p.hpg == 1 && p.ndir == 1) return false;
  const int es = p.io_dt ? 2 : 4;
  for (int d = 0; d < p.ndir; ++d) {
    const TensorD* ts[2] = {&p.x[d], &p.dout[d]};
    for (const TensorD* t : ts)
      if ((dy_ws && t == &p.dout[d]) ? (p.P & 3) != 0 : (p.P & 3) || ((t->s0 | t->s1 | t->s2) & 3) || (((uintptr_t)t->ptr) & (4 * es - 1))) return false;
  }
  return true;
}

// Whether one launch takes both directions (DUAL).  Complete tiles: only then do the two directions' chunks cover the same tokens.
// bf16, or fp32 heads of 32: others of up to 31 and of 33 to 48 spill 48 - 92 bytes a lane (8 x 1024 tokens, 8 heads x 36, 256 states,
// training step 526 us in two launches, 535 in one), and of more than 48 lose at five barriers a head what the traffic saves (16 x 2048
// tokens, 16 heads x 64, 512 states: the kernel 3.60 and 3.59 ms).  From 321 workgroups on: a workgroup fills a CU, so up to 256 leave CUs
// idle and a few more need another round (320 of them, fp32: 333 against 335 us; 384: 371 and 369; 576: 583 and 562).
bool bwd_tile_dual(const KP& p, const float* dy_ws, int parts) {
  const long blocks = (long)p.B * p.nc * p.G * ((p.N + NS - 1) / NS);
  return p.ndir == 2 && p.full_tiles && !dy_ws && parts == 1 && blocks > 320 && (p.io_dt || p.P == 32) && bwd_tile_available(p, dy_ws);
}

// Whether two heads of a group share a workgroup (PAIR): an even number of them, in calls of one direction, where no CU gets a second
// workgroup: two waves a SIMD then take half as many heads each.  Against two workgroups that share the heads (PARTS) it saves
// the launch that adds up their sums: 4 x 1024 tokens, 8 heads x 32, 256 states, fp32 45.2 + 6.9 us -> 44.0, bf16 35.6 + 7.2 -> 34.0; heads of 64
// 58.2 + 6.8 -> 60.0; three parts, 3 x 1024, fp32 42.6 + 6.3 -> 42.0, heads of 36, bf16 36.4 + 6.2 -> 37.0.
static bool bwd_tile_pair(const KP& p, int blocks, int parts) { return p.ndir == 1 && parts == 1 && blocks <= NCU && p.hpg % 2 == 0; }

template <int PT, bool IOB>
static int launch_bwd_tile_t(const KP& p, int blocks, const float* states, const float* dstates, const float* dm,
                             float* partA, float* partBias, int* redo, int parts, bool dual, DxPart dx, int dx_blocks, hipStream_t st) {
  static_assert(sizeof(BwdTileSmem<PT, !IOB>) <= 80 * 1024, "two workgroups a CU");
  const bool pnf = p.P == 16 * PT, acc = p.dir0 > 0, pair = bwd_tile_pair(p, blocks, parts);
  auto go = [&](auto kern, int dirs = 1) -> int {
    typedef BwdTileSmem<PT, !IOB> SM;
    const size_t sm = pair ? std::max(2 * sizeof(SM), sizeof(BwdDxSmem<PT, IOB, 2>)) : dirs == 1 ? sizeof(SM) : dual_lds<SM>();
    if (sm > 64 * 1024)
      if (int e = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm))
        return e;
    hipLaunchKernelGGL(kern, dim3(blocks + dx_blocks, parts), dim3(dirs * NTHREADS), sm, st, p, states, dstates, dm, partA, partBias, redo,
                       pair ? p.hpg / 2 : (p.hpg + parts - 1) / parts, dx);
    return 0;
  };
  if constexpr (IOB)
    if (dual && !pnf) return go(&k_bwd_tile<DUAL_TILES + PT, IOB, false, false, false, true, false>, 2);
  if constexpr (IOB || PT == 2)
    if (dual) return go(&k_bwd_tile<DUAL_TILES + PT, IOB, true, false, false, true, false>, 2);
  if (pair) {
    if (!p.full_tiles) return go(&k_bwd_tile<PAIR_TILES + PT, IOB, false, false, false, false, false>, 2);
    if (pnf) return go(&k_bwd_tile<PAIR_TILES + PT, IOB, true, false, false, true, false>, 2);
    return go(&k_bwd_tile<PAIR_TILES + PT, IOB, false, false, false, true, false>, 2);
  }
  auto pick = [&](auto p32) -> int {
    constexpr bool P32 = decltype(p32)::value;
    if (parts > 1) {
      if (!p.full_tiles) return acc ? go(&k_bwd_tile<PT, IOB, false, true, P32, false, true>) : go(&k_bwd_tile<PT, IOB, false, false, P32, false, true>);
      return acc ? go(&k_bwd_tile<PT, IOB, false, true, P32, true, true>) : go(&k_bwd_tile<PT, IOB, false, false, P32, true, true>);
    }
    if (!p.full_tiles) return acc ? go(&k_bwd_tile<PT, IOB, false, true, P32, false, false>) : go(&k_bwd_tile<PT, IOB, false, false, P32, false, false>);
    if (pnf) return acc ? go(&k_bwd_tile<PT, IOB, true, true, P32, true, false>) : go(&k_bwd_tile<PT, IOB, true, false, P32, true, false>);
    return acc ? go(&k_bwd_tile<PT, IOB, false, true, P32, true, false>) : go(&k_bwd_tile<PT, IOB, false, false, P32, true, false>);
  };
  if constexpr (IOB)
    if (p.ddt_part.ptr) return pick(std::true_type{});
  return pick(std::false_type{});
}

int launch_bwd_tile(const KP& p_, const float* dy_ws, const float* states, const float* dstates, const float* dm,
                    float* partA, float* partBias, int* redo, int parts, bool dual, const float* cabt, float* partD, bool* with_dx,
                    hipStream_t st) {
  KP p = p_;
  if (dy_ws) {  // a gated dy: fp32 (Bt, L, H, P) contiguous, batch * direction outermost
    TensorD& t = p.dout[p.dir0];
    t.s2 = p.P;
    t.s1 = (long)p.H * p.P;
    t.s0 = (long)p.ndir * p.L * p.H * p.P;
    t.ptr = dy_ws + (long)p.dir0 * p.L * p.H * p.P;
    p.full_tiles = 0;   // the variants with fp32 products, see the head of this file
  }
  const int blocks = p.B * p.nc * p.G * ((p.N + NS - 1) / NS);
  const int pt = (p.P + 15) / 16, units = p.B * p.nc * p.H;
  // dx beside it: a CU for each workgroup of either (and two slices of the states, which dx's two groups of waves share)
  const bool dx = with_dx && !dy_ws && bwd_tile_pair(p, blocks, parts) && two_groups(units, p.N) && blocks + units <= NCU;
  const DxPart dxp{cabt, partD, blocks};
  const int dxb = dx ? units : 0;
  if (with_dx) *with_dx = dx;
  int e = 0;
  if (p.io_dt) {
    if (pt <= 2) e = launch_bwd_tile_t<2, true>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
    else if (pt == 3) e = launch_bwd_tile_t<3, true>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
    else e = launch_bwd_tile_t<4, true>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
  } else {
    if (pt <= 2) e = launch_bwd_tile_t<2, false>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
    else if (pt == 3) e = launch_bwd_tile_t<3, false>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
    else e = launch_bwd_tile_t<4, false>(p, blocks, states, dstates, dm, partA, partBias, redo, parts, dual, dxp, dxb, st);
  }
  if (e) return e;
  return (int)hipGetLastError();
}

}  // namespace issm
