// Point-set operators of the PointNet++ backbone for gfx950: furthest point sampling, ball query, grouping,
// gathering, 3-nearest-neighbour search and interpolation (the functions of the reference's `pointnet2._ext`,
// pointnet2/_ext_src/src/*.cpp).  Index arithmetic is exact; all tensors fp32 / int32, contiguous.
//
//  * furthest point sampling: one workgroup per sample; up to 24576 points live in registers with their running minimum
//    distance, sorted into groups of 64 neighbours so that a draw looks only at groups it can change; beyond that
//    coordinates are re-read and distances kept in the caller's `temp`.  Ties go to the smaller index.
//  * ball query: points are tested in index order, 64 a step, until a centre has its `nsample` hits; balls too empty for that
//    are found through masks of the centres near an interval of each axis.
//  * 3-NN: one thread per unknown point; 256 to 8192 known points are sorted into a grid in LDS of which a thread looks at
//    the cells around its point, fewer or more are staged through LDS 256 at a time and all looked at.
//  * group / interpolate and their gradients: whole rows (one channel's points) live in LDS, the indices of a sample stream
//    past them; gradients are summed there and written once.  Rows too long for LDS, and gathers of fewer entries than a
//    row has points, take one thread per output element; their gradients scatter with hardware float atomics -- either
//    straight into the (b, c, n) layout, one scattered cache line per lane, or (the *_cl entry points) into a channel-last
//    (b, n, c) buffer through an LDS transpose, 64 consecutive floats per instruction.
#include <algorithm>
#include <type_traits>

#include "issm_dev.h"

namespace issm {

constexpr int ROW_POINTS = 40960;     // points of a row that fit in a CU's 160 KB of LDS
constexpr int INTERP_POINTS = 10240;  // of four rows
constexpr int WIDE_POINTS = 5120;     // of a row of doubles, four workgroups to a CU

constexpr int FPS_T = 512;    // threads of the sampling workgroup (two waves per SIMD: 256 registers each)

// Squared distance in plain fp32 steps (three subtractions, three products, two additions, each rounded): no fused
// multiply-add and no reordering, so the comparisons that pick indices agree with a straightforward fp32 evaluation.
__device__ __forceinline__ float sqdist(float ax, float ay, float az, float bx, float by, float bz) {
#pragma clang fp contract(off) reassociate(off)
  const float dx = ax - bx, dy = ay - by, dz = az - bz;
  const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
  return (xx + yy) + zz;
}

struct ArgMax {
  float v;
  int i;
};
__device__ __forceinline__ ArgMax better(ArgMax a, ArgMax b) {  // larger value, then smaller index
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

// idxs[b][0] = 0; then repeatedly the point farthest from the chosen set.  Points with |p|^2 <= 1e-3 (padding at the
// origin) are never chosen and keep their distance, as in the reference (sampling_gpu.cu:105-106).

// Wave-wide maxima with DPP: four shifts inside each row of 16 lanes, then the rows (zero, what lanes without a source
// receive, is the identity of an unsigned maximum, so a step is one v_max_u32).
__device__ __forceinline__ unsigned umax(unsigned a, unsigned b) { return a > b ? a : b; }
__device__ __forceinline__ unsigned umin(unsigned a, unsigned b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }
__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
#define UMAX_STEP(ctrl) v = umax(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xf, 0xf, true))
// the maximum over the first ROWS * 16 lanes (ROWS = 1, 2 or 4), in a scalar register
template <int ROWS>
__device__ __forceinline__ unsigned wave_max(unsigned v) {
  UMAX_STEP(0x111); UMAX_STEP(0x112); UMAX_STEP(0x114); UMAX_STEP(0x118);
  if (ROWS >= 2) v = umax(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row 0 -> 1, 2 -> 3
  if (ROWS == 4) v = umax(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row 1 -> 2, 3
  return (unsigned)__builtin_amdgcn_readlane((int)v, 16 * ROWS - 1);
}
#undef UMAX_STEP
__device__ __forceinline__ float wave_fmax(float v) {  // (used once per slot, not per draw)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float lane_f(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
// of the lanes in `cand`, the one with the smallest `key` (equal distances; keys differ).  One reduction however many there
// are: on a voxelized cloud most lanes tie, and taken one by one they made a draw three times as long (8192 points on a
// quarter-metre grid, 2048 draws, 8 samples: 6.9 -> 2.2 ms).
__device__ __forceinline__ int lane_of_least(unsigned long long cand, int key) {
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const unsigned v = (cand >> lane) & 1ull ? ~(unsigned)key : 0u;   // keys are >= 0, so a candidate's v is never 0
  const unsigned m = wave_max<4>(v);
  return __builtin_ctzll(__ballot(v == m));
}

// Up to 64 W S points: one workgroup of W waves per sample, points in registers, and only those looked at that a draw can
// change.  The draws are a serial chain, so what counts is the time of one: passing over all points costs 40 distances
// per lane at 20000 points (1.92 us a draw, the vector unit of one CU saturated).  Here the points are first sorted along a
// Z-order curve over a 16^3 grid (counting sort in LDS) and cut into groups of 64 neighbours, one point per lane; group g
// belongs to wave g % W (neighbouring groups to different waves) as its slot g / W, and lane l of the wave keeps slot l's
// bounding box, largest running distance and the point that has it.  A draw at o compares o's distance to every box with
// the group's largest distance -- one instruction sequence for all groups of a wave -- and goes through the points of
// those groups only that are nearer: about 15 of 313.  Few of these lose their farthest point: where that one is as far as
// before, the group's best is what it was, and a wave none of whose groups has another best hands over the same one again.
// One barrier per draw (the waves' bests go through LDS buffers used in turn).  20000 points, 2048 draws, 8 samples: 3.93 ms
// looking at all points, 1.94 looking for the best of every group gone through, 1.55 here (0.57 us a draw of a chain through
// a reduction over a group, one over a wave's groups, LDS, a barrier and one over the waves, the rest the groups looked at).
//
// The pruning is exact: fp32 rounding is monotone, so for a point q of the box each step of the box's squared distance
// (subtract, square, add, in sqdist's order) is at most the same step for q, and where the box's distance is not below the
// group's largest running distance, no minimum of the group changes.  A NaN anywhere makes the comparison fail, which means
// "look".  Equal distances go to the smaller index at every level, as a pass over all points in order would decide.
//
// What the pruning saves depends on how small the groups' boxes are, so the grid must fit the cloud: one point 300 m away from
// a room of 8 m would leave the room a single cell of a grid over everything, its groups in index order and every box the
// whole room.  The grid therefore covers what most points fill -- the middle half of a sample along each axis and as much again
// on either side -- and a second, coarser one, sorted behind it, everything.  20000 points, 2048 draws, 8 samples: uniform 1.95
// ms; with one far point 9.5 -> 1.97, one in twenty far 5.5 -> 1.88, a third far 1.77 -> 1.73 (passing over all points: 3.9), all
// before bests were kept: 1.56, 1.67, 1.53 and 1.41 with that.
constexpr int FPS_CELLS = 4096, FPS_BINS = 5120;   // 16^3 cells and 8^3 behind them, rounded up to a multiple of the threads
// f(0), f(1), ... f(N - 1) with constant arguments: register arrays indexed inside f stay in registers for every N (the
// loop unroller left a loop over 20 or 24 slots to dynamic indexing, and the arrays to scratch)
template <int N, int I = 0, class F>
__device__ __forceinline__ void for_each_slot(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    for_each_slot<N, I + 1>(static_cast<F&&>(f));
  }
}
__device__ __forceinline__ unsigned spread4(unsigned v) {   // bits 0..3 -> 0, 3, 6, 9
  return (v & 1u) | ((v & 2u) << 2) | ((v & 4u) << 4) | ((v & 8u) << 6);
}

template <int W, int S>
__global__ __launch_bounds__(64 * W) void k_fps_groups(int n, int npoint, const float* __restrict__ xyz, int* __restrict__ idxs) {
  constexpr int T = 64 * W, ROWS = (S + 15) / 16;
  static_assert(S % 4 == 0 && S <= 32 && W <= 16 && (W & (W - 1)) == 0, "slots and waves sit in the lanes of one wave");
  __shared__ int hist[FPS_BINS];
  __shared__ unsigned short order[T * S];
  __shared__ float quart[6];
  __shared__ int sampled;
  __shared__ float red[6][W];
  __shared__ int wsum[W];
  struct alignas(16) Best { unsigned d; float x, y, z; };
  __shared__ Best best[2][W];
  __shared__ int best_pos[2][W];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* p = xyz + (long)b * n * 3;
  int* out = idxs + (long)b * npoint;
  const float INFV = __builtin_huge_valf();

  // quartiles of a sample of 64 points: wave a takes axis a, a lane counts the values before its own
  if (wave < 3) {
    const float* q = p + (long)lane * n / 64 * 3;
    const float x = q[0], y = q[1], z = q[2], r = sqdist(x, y, z, 0.0f, 0.0f, 0.0f);
    const float v = r > 1e-3f && r < INFV ? (wave == 0 ? x : wave == 1 ? y : z) : INFV;
    const int m = __popcll(__ballot(v < INFV));
    int before = 0;
#pragma unroll 8
    for (int j = 0; j < 64; ++j) {
      const float u = lane_f(v, j);
      before += u < v || (u == v && j < lane) ? 1 : 0;
    }
    if (before == m / 4) quart[wave] = v;
    if (before == m - 1 - m / 4) quart[3 + wave] = v;
    if (tid == 0) sampled = m;
  }
  // bounding box of the points that take part
  float lo[3] = {INFV, INFV, INFV}, hi[3] = {-INFV, -INFV, -INFV};
  for (int k = tid; k < n; k += T) {
    const float x = p[k * 3], y = p[k * 3 + 1], z = p[k * 3 + 2];
    if (sqdist(x, y, z, 0.0f, 0.0f, 0.0f) > 1e-3f) {
      lo[0] = fminf(lo[0], x); lo[1] = fminf(lo[1], y); lo[2] = fminf(lo[2], z);
      hi[0] = fmaxf(hi[0], x); hi[1] = fmaxf(hi[1], y); hi[2] = fmaxf(hi[2], z);
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float l = -wave_fmax(-lo[a]), h = wave_fmax(hi[a]);
    if (lane == 0) { red[a][wave] = l; red[3 + a][wave] = h; }
  }
  for (int c = tid; c < FPS_BINS; c += T) hist[c] = 0;
  __syncthreads();
  float ext = 0.0f, ext1 = 0.0f, lo1[3], hi1[3];   // 1: of the grid over most points
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    for (int w = 0; w < W; ++w) { lo[a] = fminf(w ? lo[a] : INFV, red[a][w]); hi[a] = fmaxf(w ? hi[a] : -INFV, red[3 + a][w]); }
    ext = fmaxf(ext, hi[a] - lo[a]);
    const float half = quart[3 + a] - quart[a];
    lo1[a] = sampled < 8 ? lo[a] : fmaxf(lo[a], quart[a] - half);
    hi1[a] = sampled < 8 ? hi[a] : fminf(hi[a], quart[3 + a] + half);
    ext1 = fmaxf(ext1, hi1[a] - lo1[a]);
  }
  const float inv = ext > 0.0f && ext < INFV ? 8.0f / ext : 0.0f, inv1 = ext1 > 0.0f && ext1 < INFV ? 16.0f / ext1 : 0.0f;
  auto cell = [&](int k) {
    const float v[3] = {p[k * 3], p[k * 3 + 1], p[k * 3 + 2]};
    bool most = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) most = most && v[a] >= lo1[a] && v[a] <= hi1[a];
    unsigned c = most ? 0 : FPS_CELLS;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      c |= spread4((unsigned)imin(imax((int)((v[a] - (most ? lo1[a] : lo[a])) * (most ? inv1 : inv)), 0), most ? 15 : 7)) << a;
    return c;
  };
  for (int k = tid; k < n; k += T) atomicAdd(&hist[cell(k)], 1);
  __syncthreads();
  {  // exclusive prefix sum of the histogram: FPS_BINS / T neighbours per thread
    constexpr int E = FPS_BINS / T;
    int own = 0;
    for (int e = 0; e < E; ++e) own += hist[tid * E + e];
    int incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int at = incl - own;
    for (int w = 0; w < wave; ++w) at += wsum[w];
    for (int e = 0; e < E; ++e) { const int v = hist[tid * E + e]; hist[tid * E + e] = at; at += v; }
  }
  __syncthreads();
  for (int k = tid; k < n; k += T) order[atomicAdd(&hist[cell(k)], 1)] = (unsigned short)k;
  __syncthreads();

  // the wave's slots into registers; lane l keeps what belongs to slot l.  A running distance is kept as its bit pattern
  // plus one: distances are >= 0 and order as unsigned integers do, 0 marks a point that never takes part (or a lane
  // without a slot), and a NaN or infinite distance is above every running one.
  const unsigned far = __builtin_bit_cast(unsigned, 1e10f) + 1u;
  float px[S], py[S], pz[S];
  unsigned d[S];
  float blx = INFV, bly = INFV, blz = INFV, bhx = -INFV, bhy = -INFV, bhz = -INFV, gx = 0.0f, gy = 0.0f, gz = 0.0f;
  unsigned gd = 0;
  int gpos = 0;
  for_each_slot<S>([&](auto slot) {
    constexpr int j = decltype(slot)::value;
    const int pos = (j * W + wave) * 64 + lane;
    px[j] = py[j] = pz[j] = 0.0f;
    if (pos < n) { const int k = order[pos]; px[j] = p[k * 3]; py[j] = p[k * 3 + 1]; pz[j] = p[k * 3 + 2]; }
    const bool in = sqdist(px[j], py[j], pz[j], 0.0f, 0.0f, 0.0f) > 1e-3f;
    d[j] = in ? far : 0u;
    const float lx = -wave_fmax(in ? -px[j] : -INFV), ly = -wave_fmax(in ? -py[j] : -INFV), lz = -wave_fmax(in ? -pz[j] : -INFV);
    const float hx = wave_fmax(in ? px[j] : -INFV), hy = wave_fmax(in ? py[j] : -INFV), hz = wave_fmax(in ? pz[j] : -INFV);
    const unsigned long long members = __ballot(in);
    // the group's best until a draw changes it: all members are equally far, so the smallest index.  (A group whose box is
    // `far` or more from every draw is never looked at -- points 1e5 apart, infinite coordinates -- and is chosen as it is.)
    const int l = lane_of_least(members, pos < n ? (int)order[pos] : 0x7fffffff);
    const float x = lane_f(px[j], l), y = lane_f(py[j], l), z = lane_f(pz[j], l);
    if (lane == j) {
      blx = lx; bly = ly; blz = lz; bhx = hx; bhy = hy; bhz = hz;
      gd = members ? far : 0u;
      gpos = (j * W + wave) * 64 + l;
      gx = x; gy = y; gz = z;
    }
  });
  float ox = p[0], oy = p[1], oz = p[2];
  bool changed = true;   // (uniform) one of the wave's groups has another best since the wave's best was looked for
  int mine = 0;          // the slot with the wave's best
  for (int s = 1; s < npoint; ++s) {
    // the slots whose box is nearer than their largest distance (never NaN: fmaxf drops one)
    const float ex = fmaxf(fmaxf(blx - ox, ox - bhx), 0.0f), ey = fmaxf(fmaxf(bly - oy, oy - bhy), 0.0f),
                ez = fmaxf(fmaxf(blz - oz, oz - bhz), 0.0f);
    const unsigned mask = (unsigned)__ballot(__builtin_bit_cast(unsigned, sqdist(ex, ey, ez, 0.0f, 0.0f, 0.0f)) + 1u < gd);
    for_each_slot<S / 4>([&](auto block) {
      constexpr int j4 = 4 * decltype(block)::value;
      if (((mask >> j4) & 15u) == 0) return;
      for_each_slot<4>([&](auto slot) {
        constexpr int j = j4 + decltype(slot)::value;
        if (((mask >> j) & 1u) == 0) return;
        const unsigned before = (unsigned)__builtin_amdgcn_readlane((int)gd, j);
        const int at = __builtin_amdgcn_readlane(gpos, j) & 63;
        d[j] = umin(d[j], __builtin_bit_cast(unsigned, sqdist(px[j], py[j], pz[j], ox, oy, oz)) + 1u);
        if ((__ballot(d[j] == before) >> at) & 1ull) return;   // its best is as far as before, and no other point is farther
        const unsigned m = wave_max<4>(d[j]);
        const unsigned long long cand = __ballot(d[j] == m);
        const int base = (j * W + wave) * 64;
        int l = __builtin_ctzll(cand);
        if (__builtin_expect(__popcll(cand) > 1, 0)) l = lane_of_least(cand, base + lane < n ? (int)order[base + lane] : 0x7fffffff);
        const float x = lane_f(px[j], l), y = lane_f(py[j], l), z = lane_f(pz[j], l);
        if (lane == j) { gd = m; gpos = base + l; gx = x; gy = y; gz = z; }
        changed = true;
      });
    });
    // the wave's best, then the workgroup's
    if (changed) {
      const unsigned m = wave_max<(S > 16 ? 2 : 1)>(gd);
      const unsigned long long cand = __ballot(gd == m);
      mine = __builtin_ctzll(cand);
      if (__builtin_expect(__popcll(cand) > 1, 0) && m) mine = lane_of_least(cand, (int)order[gpos]);
      changed = false;
    }
    if (lane == mine) { best[s & 1][wave] = Best{gd, gx, gy, gz}; best_pos[s & 1][wave] = gpos; }
    __syncthreads();
    Best w = best[s & 1][lane & (W - 1)];   // repeated through the wave: the first row holds every wave's
    const int wp = best_pos[s & 1][lane & (W - 1)];
    const unsigned m = wave_max<1>(w.d);
    const unsigned cand = (unsigned)__ballot(w.d == m) & ((1u << W) - 1);
    int l = __builtin_ctz(cand);
    bool none = false;
    if (__builtin_expect(__popc(cand) > 1, 0)) {   // (all waves, if nothing but padding points is left)
      none = m == 0;
      if (!none) l = lane_of_least(cand, (int)order[wp]);
    }
    ox = lane_f(w.x, l); oy = lane_f(w.y, l); oz = lane_f(w.z, l);
    if (__builtin_expect(none, 0)) { ox = p[0]; oy = p[1]; oz = p[2]; }   // index 0, as the reference
    if (tid == l) out[s] = none ? -1 : wp;   // a place in `order` for now: its translation would be waited for here
  }
  __syncthreads();
  for (int s = tid; s < npoint; s += T) out[s] = s && out[s] >= 0 ? (int)order[out[s]] : 0;
}

// Any number of points (used above 24576, where they no longer fit one workgroup's registers): coordinates re-read from
// memory (L2) and distances kept in `temp`.
__global__ __launch_bounds__(FPS_T) void k_fps(int n, int npoint, const float* __restrict__ xyz, float* __restrict__ temp,
                                                int* __restrict__ idxs) {
  __shared__ float sv[FPS_T / 64];
  __shared__ int si[FPS_T / 64];
  __shared__ int chosen;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* p = xyz + (long)b * n * 3;
  int* out = idxs + (long)b * npoint;
  float* tmp = temp + (long)b * n;
  for (int k = tid; k < n; k += FPS_T) tmp[k] = 1e10f;
  if (tid == 0) out[0] = 0;
  int old = 0;
  for (int s = 1; s < npoint; ++s) {
    const float ox = p[old * 3], oy = p[old * 3 + 1], oz = p[old * 3 + 2];
    float bv = -1.0f;
    int bi = 0;
    for (int k = tid; k < n; k += FPS_T) {
      const float x = p[k * 3], y = p[k * 3 + 1], z = p[k * 3 + 2];
      if (sqdist(x, y, z, 0.0f, 0.0f, 0.0f) > 1e-3f) {
        const float d = fminf(tmp[k], sqdist(x, y, z, ox, oy, oz));
        tmp[k] = d;
        if (d > bv) { bv = d; bi = k; }
      }
    }
    ArgMax best = {bv, bi};
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ArgMax other = {__shfl_xor(best.v, o, 64), __shfl_xor(best.i, o, 64)};
      best = better(best, other);
    }
    if (lane == 0) { sv[wave] = best.v; si[wave] = best.i; }
    __syncthreads();
    if (tid == 0) {
      ArgMax a = {sv[0], si[0]};
      for (int w = 1; w < FPS_T / 64; ++w) a = better(a, ArgMax{sv[w], si[w]});
      chosen = a.v > -1.0f ? a.i : 0;  // nothing but padding points: index 0, as the reference
      out[s] = chosen;
    }
    __syncthreads();
    old = chosen;
  }
}

// idx[b][j][0..nsample): the first nsample points (in index order) closer than radius to new_xyz[b][j]; missing
// slots repeat the first hit; no hit at all leaves zeros (ball_query_gpu.cu:20-44).
//
// A workgroup takes 64 centres, and what it does for one depends on how many points the first BQ_PREFIX show its ball to have.
// Full balls are found by looking at points in order, 64 a step and four centres a wave, until a centre has nsample hits (its
// wave compacts them in index order with a ballot).  The others would look at many points in vain: for them the axes are cut
// into 64 intervals each, whose 64-bit masks name the centres with an interval within the radius; a thread takes a point, ANDs
// the three masks of its place and tests the few centres that are left.  Their hits come in any order, into lists in LDS, and
// are put in order by counting; a centre that has enough after a chunk of points leaves the masks, and one whose list overflows
// within a chunk (BQ_CAP) keeps what it had before and looks at points in order from there.
// The masks leave out no hit: rounding is monotone, so a distance below the radius means a coordinate within [q - r, q + r] as
// these are rounded, and the interval's number is a monotone function of the coordinate (a coordinate that is no number, or
// a grid without extent, is interval 0).
// Bound by the passes over the points.  8 samples, 2048 centres, 20000 points in a room of 8 m, 64 slots, against one centre a
// wave and every point in order: radius 0.2 229 -> 26 us; calls with radius 0.8 165 -> 48, 1.2 107 -> 62; one sample, 512
// centres: 69 -> 19, 69 -> 25, 61 -> 29.
constexpr int BQ_T = 1024, BQ_CAP = 128, BQ_PREFIX = 1024, BQ_CHUNK = 4 * BQ_T;
template <int EACH>   // centres of a wave
__global__ __launch_bounds__(BQ_T) void k_ball_query(int n, int m, float radius, float radius2, int nsample,
                                                     const float* __restrict__ new_xyz, const float* __restrict__ xyz,
                                                     int* __restrict__ idx) {
  constexpr int CENTRES = EACH * (BQ_T / 64);
  static_assert(CENTRES <= 64 && BQ_CAP == 128, "a bit of a mask for each, two hits of a list a lane");
  __shared__ float centre[3][CENTRES];
  __shared__ unsigned long long bits[3][64];
  __shared__ float from[3], scale[3];
  __shared__ unsigned long long listed;       // the centres that take the masks
  __shared__ int count[CENTRES];
  __shared__ __align__(16) int list[CENTRES][BQ_CAP];
  __shared__ int need[CENTRES], kept[CENTRES], resume[CENTRES];   // hits to find; hits of the list that count; where to go on
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j0 = blockIdx.x * CENTRES;
  const float* p = xyz + (long)b * n * 3;
  if (tid < CENTRES) {
    const float* q = new_xyz + ((long)b * m + min(j0 + tid, m - 1)) * 3;
#pragma unroll
    for (int a = 0; a < 3; ++a) centre[a][tid] = q[a];
    count[tid] = kept[tid] = 0;
    resume[tid] = n;
    if (tid == 0) listed = 0;
  }
  __syncthreads();
  // the wave's centres: hits so far, the first of them
  float qx[EACH], qy[EACH], qz[EACH];
  int cnt[EACH], first[EACH];
  unsigned todo = 0;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int c = wave * EACH + i;
    qx[i] = centre[0][c]; qy[i] = centre[1][c]; qz[i] = centre[2][c];
    cnt[i] = first[i] = 0;
    if (j0 + c < m && nsample > 0) todo |= 1u << i;
  }
  int* out = idx + ((long)b * m + j0 + wave * EACH) * nsample;
  // points lo .. hi - 1 in order, for the centres in `todo`; those that have nsample hits leave it
  auto look = [&](int lo, int hi, unsigned todo) {
    for (int k0 = lo; k0 < hi && todo; k0 += 256) {
      float x[4], y[4], z[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* q = p + (long)min(k0 + 64 * u + lane, n - 1) * 3;
        x[u] = q[0]; y[u] = q[1]; z[u] = q[2];
      }
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        if (!(todo >> i & 1u)) continue;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = k0 + 64 * u + lane;
          const bool hit = k < hi && sqdist(qx[i], qy[i], qz[i], x[u], y[u], z[u]) < radius2;
          const unsigned long long mask = __ballot(hit);
          if (mask == 0) continue;
          if (cnt[i] == 0) first[i] = k0 + 64 * u + __builtin_ctzll(mask);
          const int slot = cnt[i] + __popcll(mask & ((1ull << lane) - 1ull));
          if (hit && slot < nsample) out[i * nsample + slot] = k;
          cnt[i] += __popcll(mask);
        }
        if (cnt[i] >= nsample) todo &= ~(1u << i);
      }
    }
    return todo;
  };
  const int prefix = min(n, BQ_PREFIX);
  todo = look(0, prefix, todo);
  unsigned sparse = 0;
  if (prefix < n) {
#pragma unroll
    for (int i = 0; i < EACH; ++i)
      if ((todo >> i & 1u) && cnt[i] * (BQ_CHUNK / BQ_PREFIX) + min(nsample, BQ_CAP / 2) <= BQ_CAP && nsample - cnt[i] > 2 * cnt[i]) {
        sparse |= 1u << i;
        if (lane == 0) need[wave * EACH + i] = nsample - cnt[i];
      }
    if (sparse && lane == 0) atomicOr(&listed, (unsigned long long)sparse << (wave * EACH));
  } else {
    todo = 0;
  }
  __syncthreads();
  const unsigned long long those = listed;
  if (those) {   // uniform
    const float r = fabsf(radius);
    if (wave < 3) {   // an axis each
      const float q = centre[wave][lane & (CENTRES - 1)], qlo = q - r, qhi = q + r;
      const bool in = those >> lane & 1ull;
      const float lo = -wave_fmax(in ? -qlo : -__builtin_huge_valf()), hi = wave_fmax(in ? qhi : -__builtin_huge_valf());
      const float ext = hi - lo, inv = ext > 0.0f ? 64.0f / ext : 0.0f;
      const int c0 = min(max((int)((qlo - lo) * inv), 0), 63), c1 = min(max((int)((qhi - lo) * inv), 0), 63);
      unsigned long long own = 0;
      for (int e = 0; e < 64; ++e) {
        const unsigned long long mask = __ballot(in && c0 <= e && e <= c1);
        if (lane == e) own = mask;
      }
      bits[wave][lane] = own;
      if (lane == 0) { from[wave] = lo; scale[wave] = inv; }
    }
    __syncthreads();
    const float lo0 = from[0], lo1 = from[1], lo2 = from[2], s0 = scale[0], s1 = scale[1], s2 = scale[2];
    auto interval = [&](float v, float lo, float s) { return min(max((int)((v - lo) * s), 0), 63); };
    constexpr int U = BQ_CHUNK / BQ_T;
    unsigned long long active = those;   // (in every thread)
    for (int k0 = prefix; k0 < n && active; k0 += BQ_CHUNK) {
      float x[U], y[U], z[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* q = p + (long)min(k0 + BQ_T * u + tid, n - 1) * 3;
        x[u] = q[0]; y[u] = q[1]; z[u] = q[2];
      }
      unsigned long long near[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        near[u] = bits[0][interval(x[u], lo0, s0)] & bits[1][interval(y[u], lo1, s1)] & bits[2][interval(z[u], lo2, s2)] & active;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + BQ_T * u + tid;
        if (k >= n) near[u] = 0;
        while (near[u]) {
          const int c = __builtin_ctzll(near[u]);
          near[u] &= near[u] - 1;
          if (sqdist(centre[0][c], centre[1][c], centre[2][c], x[u], y[u], z[u]) < radius2) {
            const int at = atomicAdd(&count[c], 1);
            if (at < BQ_CAP) list[c][at] = k;
          }
        }
      }
      __syncthreads();
      const int found = count[lane & (CENTRES - 1)];   // every wave for itself (lanes beyond the centres are not in `active`)
      const bool over = found > BQ_CAP;
      const unsigned long long leave = __ballot(over || found >= need[lane & (CENTRES - 1)]) & active;
      if (wave == 0 && (active >> lane & 1ull)) {
        if (over) resume[lane] = k0;
        else kept[lane] = found;
      }
      active &= ~leave;
      __syncthreads();   // (count is read before the next chunk adds to it)
    }
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      if (!(sparse >> i & 1u)) continue;
      const int c = wave * EACH + i, found = __builtin_amdgcn_readfirstlane(kept[c]);
      if (found) {
        const int none = 0x7fffffff, e0 = lane < found ? list[c][lane] : none, e1 = 64 + lane < found ? list[c][64 + lane] : none;
        int r0 = cnt[i], r1 = cnt[i];
        for (int t0 = 0; t0 < found; t0 += 8) {   // (BQ_CAP is a multiple of 8: what is read behind the hits lies in the list)
          const int4 va = *(const int4*)&list[c][t0], vb = *(const int4*)&list[c][t0 + 4];
          const int v[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int w = t0 + j < found ? v[j] : none;
            r0 += w < e0 ? 1 : 0;
            r1 += w < e1 ? 1 : 0;
          }
        }
        if (e0 != none && r0 < nsample) out[i * nsample + r0] = e0;
        if (e1 != none && r1 < nsample) out[i * nsample + r1] = e1;
        if (cnt[i] == 0) {
          const unsigned long long f0 = __ballot(e0 != none && r0 == 0), f1 = __ballot(e1 != none && r1 == 0);
          first[i] = f0 ? __builtin_amdgcn_readlane(e0, __builtin_ctzll(f0)) : __builtin_amdgcn_readlane(e1, __builtin_ctzll(f1));
        }
        cnt[i] += found;
      }
    }
#pragma unroll
    for (int i = 0; i < EACH; ++i)
      if (sparse >> i & 1u) look(__builtin_amdgcn_readfirstlane(resume[wave * EACH + i]), n, 1u << i);
    todo &= ~sparse;
  }
  look(prefix, n, todo);
#pragma unroll
  for (int i = 0; i < EACH; ++i)
    if (j0 + wave * EACH + i < m)
      for (int s = min(cnt[i], nsample) + lane; s < nsample; s += 64) out[i * nsample + s] = first[i];  // (0 if nothing was found)
}

// Grouping.  Output channel ch < cx (cx = 0 or 3): coordinate ch of the point relative to the entry's centre, times `scale`;
// then the c feature channels.
struct GroupP {
  int c, cx, n, ms, npoints, nsample, rows;   // rows: of the whole batch
  long share;
  const float *xyz, *centre, *points;
  const int* idx;
  float* out;
  float scale;
};
__device__ __forceinline__ int index_of(int v, int n) { return min(max(v, 0), n - 1); }  // a stray index must not leave the tensor
struct __attribute__((packed, aligned(4))) I4Any {
  int v[4];
};
// Values read or written once, past the caches' replacement order: the indices, read again for every row, stay in L2.
typedef float f4_stream __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4 ld_stream(const float* q) { return __builtin_nontemporal_load((const f4_stream*)q); }
__device__ __forceinline__ void st_stream(float* q, f4 v) { __builtin_nontemporal_store((f4_stream)v, (f4_stream*)q); }

// One thread per output element.
__global__ __launch_bounds__(NTHREADS) void k_group_points(GroupP g) {
  const int e = blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= g.ms) return;
  const int rows = g.cx + g.c;
  for (int row = blockIdx.y; row < g.rows; row += gridDim.y) {
    const int b = row / rows, ch = row % rows;
    const int k = index_of(g.idx[(long)b * g.ms + e], g.n);
    float v;
    if (ch < g.cx) v = (g.xyz[((long)b * g.n + k) * 3 + ch] - g.centre[((long)b * g.npoints + e / g.nsample) * 3 + ch]) * g.scale;
    else v = g.points[((long)b * g.c + ch - g.cx) * g.n + k];
    g.out[(long)row * g.ms + e] = v;
  }
}

// The output's entries, row after row, in equal shares of one workgroup each; of every row it meets, a workgroup holds the
// n source values in LDS and streams the indices past them, four entries per thread and step.  (A workgroup per row left a
// third of the time to the last few rows: 1048 rows on 512 places.)  The next indices are in flight while values are read and
// stored, and a row's pieces all at once: with each step waiting for its own it was latency that counted.  8 samples of 20000
// points, 131 x 131072 entries each: 243 -> 118 us, bound by writing the output (549 MB, 4.7 TB/s; 146 us with stores that
// displace the indices in L2); separate gathers, a subtraction, a product and a concatenation took 656.
__global__ __launch_bounds__(1024) void k_group_rows(GroupP g) {
  extern __shared__ float srow[];
  const int T = blockDim.x, tid = threadIdx.x, rows1 = g.cx + g.c;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);   // an XCD's workgroups: neighbouring rows, one sample's indices in its L2
  const long end = min((long)(wg + 1) * g.share, (long)g.rows * g.ms);
  for (long at = (long)wg * g.share; at < end;) {
    const int row = (int)(at / g.ms), b = row / rows1, ch = row % rows1;
    // (entries are counted without a sign: a sample has up to 2^31 - 1, and the loop steps beyond them)
    const unsigned lo = (unsigned)(at - (long)row * g.ms), hi = (unsigned)min((long)g.ms, lo + (end - at));
    at += hi - lo;
    __syncthreads();
    if (ch < g.cx) {
      const float* q = g.xyz + (long)b * g.n * 3 + ch;
      for (int k = tid; k < g.n; k += T) srow[k] = q[k * 3];
    } else {
      const float* q = g.points + ((long)b * g.c + ch - g.cx) * g.n;
      constexpr int F = 5;   // pieces in flight
      for (int k0 = 4 * tid; k0 + 3 < g.n; k0 += 4 * T * F) {
        f4 v[F];
#pragma unroll
        for (int u = 0; u < F; ++u) v[u] = ld_f4_any(q + min(k0 + 4 * T * u, g.n - 4));
#pragma unroll
        for (int u = 0; u < F; ++u)
          if (k0 + 4 * T * u + 3 < g.n) *(f4*)(srow + k0 + 4 * T * u) = v[u];
      }
      const int k = (g.n & ~3) + tid;
      if (k < g.n) srow[k] = q[k];
    }
    __syncthreads();
    const int* q = g.idx + (long)b * g.ms;
    float* o = g.out + (long)row * g.ms;
    const unsigned full = lo + ((hi - lo) & ~3u);   // four entries a thread up to here
    auto values = [&](unsigned e, const I4Any& i) {
      f4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = srow[index_of(i.v[j], g.n)];
      if (ch < g.cx) {
        // (one division per step: what a coordinate row costs beyond a feature row decides when its workgroup ends)
        const unsigned at_c = e / (unsigned)g.nsample;
        int left = (int)((at_c + 1) * g.nsample - e);
        const float* cq = g.centre + ((long)b * g.npoints + at_c) * 3 + ch;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = (v[j] - *cq) * g.scale;
          if (--left == 0 && e + j + 1 < hi) { cq += 3; left = g.nsample; }
        }
      }
      return v;
    };
    // the next step's indices are asked for before this step's values are read
    constexpr int U = 2;
    I4Any cur[U], nxt[U];
    unsigned e = lo + 4 * tid;
    if (e < full) {
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = *(const I4Any*)(q + min(e + 4 * T * u, full - 4));
    }
    for (; e < full; e += 4 * T * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) nxt[u] = *(const I4Any*)(q + min(e + 4 * T * (U + u), full - 4));
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (e + 4 * T * u < full) st_stream(o + e + 4 * T * u, values(e + 4 * T * u, cur[u]));
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = nxt[u];
    }
    if (full + tid < hi) {
      I4Any i = {};
      i.v[0] = q[full + tid];
      o[full + tid] = values(full + tid, i)[0];
    }
  }
}

// A value from the lane N places before (SHR) or after (SHL) within the row of 16 lanes; `old` where there is none.
template <int CTRL>
__device__ __forceinline__ int row_lane(int old, int v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float row_lane_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Gradient of the grouping, all of grad_points (b, c, n) written: one workgroup per channel row (and part of its entries),
// the row's n sums in LDS, grad_out streamed once.  A ball with fewer points than slots repeats its first point, and lanes
// adding to one LDS word take turns: runs of equal indices are summed first -- four consecutive entries per lane, then a
// segmented scan over the row of 16 lanes -- and only the last entry of a run adds.  How it adds decides the rest: an LDS
// float addition takes 3 cycles a lane however the words lie (measured: 0.77 lanes a nanosecond and CU), one of doubles a
// fifth of a cycle (6.4), a compare-and-swap of a word just read, if it succeeds, half a cycle.  So up to 5120 points, of
// which four workgroups still share a CU, the sums are doubles (WIDE); beyond, a lane tries one compare-and-swap and adds the
// ordinary way where another lane was faster.  A row of 2^17 entries is 2^19 bytes, and rows read from their beginnings at one
// pace ask the same memory channels at any time: every row begins at another step.  Then it is the instructions for the runs
// that count: 8 samples, 128 channels of 20000 points, 2048 balls of 64, 144 -> 126 us for those 537 MB (4.3 TB/s), whether a
// ball repeats one point or has 64 different ones (float additions alone: 152 and 677; atomics into a channel-last buffer: 495
// and 486).  2048 points, 2048 balls, 64 channels, where the next step's loads in flight count: 69 -> 53 us.  The worst for it,
// entries that hop between two points (20000 points as above): 1260 us (898; 6000).  Eight entries a lane: 159 us, the lanes'
// pieces of 32 bytes.  With splits > 1 (few rows) the parts meet in grad_points, zero before.
template <bool WIDE>
__global__ __launch_bounds__(1024) void k_group_rows_grad(int c, int c0, int cdim, int n, int ms, int splits, unsigned per,
                                                          const float* __restrict__ grad_out, const int* __restrict__ idx,
                                                          float* __restrict__ grad_points) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef typename std::conditional<WIDE, double, float>::type Sum;
  Sum* srow = reinterpret_cast<Sum*>(smem_raw);
  auto add = [&](int k, float v) {
    if constexpr (!WIDE) {
      unsigned* u = (unsigned*)srow + k;
      const unsigned e = __hip_atomic_load(u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (a volatile one is a flat load)
      if (atomicCAS(u, e, __builtin_bit_cast(unsigned, __builtin_bit_cast(float, e) + v)) == e) return;
    }
    unsafeAtomicAdd(srow + k, (Sum)v);
  };
  const int T = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wg = xcd_remap(blockIdx.x, gridDim.x), row = wg / splits, part = wg % splits, b = row / c, ch = row % c;
  for (int k = tid; k < n; k += T) srow[k] = 0;
  __syncthreads();
  const int* q = idx + (long)b * ms;
  const float* g = grad_out + ((long)b * cdim + c0 + ch) * ms;
  const unsigned hi = min((part + 1) * per, (unsigned)ms);   // (without a sign, see k_group_rows)
  auto take = [&](const I4Any& i, f4 v) {
    const bool q1 = i.v[1] == i.v[0], q2 = i.v[2] == i.v[1], q3 = i.v[3] == i.v[2];
    v[1] += q1 ? v[0] : 0.0f;
    v[2] += q2 ? v[1] : 0.0f;
    v[3] += q3 ? v[2] : 0.0f;
    // runs across lanes: s = sum of the run that ends at the lane's last entry; `on` = that run began in an earlier lane
    const bool link = row_lane<0x111>(-2, i.v[3]) == i.v[0];
    int on = q1 && q2 && q3 && link ? -1 : 0;
    float s = v[3];
    auto step = [&](auto ctrl) {
      constexpr int C = decltype(ctrl)::value;
      s += __builtin_bit_cast(float, __builtin_bit_cast(int, row_lane_f<C>(s)) & on);
      on &= row_lane<C>(0, on);
    };
    step(std::integral_constant<int, 0x111>{});
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    const float before = row_lane_f<0x111>(s), carry = link ? before : 0.0f;
    const bool end3 = row_lane<0x101>(-2, i.v[0]) != i.v[3];
    if (!q1 && i.v[0] >= 0) add(i.v[0], v[0] + carry);
    if (!q2 && i.v[1] >= 0) add(i.v[1], v[1] + (q1 ? carry : 0.0f));
    if (!q3 && i.v[2] >= 0) add(i.v[2], v[2] + (q1 && q2 ? carry : 0.0f));
    if (end3 && i.v[3] >= 0) add(i.v[3], v[3] + (q1 && q2 && q3 ? carry : 0.0f));
  };
  // a wave's steps of 256 entries, the next one's in flight, from another step on for every row; what fills no step at last
  const unsigned lo = part * per, own = lo + (tid >> 6) * 256;   // wave-uniform
  const unsigned steps = own + 256 <= hi ? (hi - own - 256) / (4 * T) + 1 : 0;
  if (steps) {
    unsigned at = row * 7u % steps;
    auto entries = [&](unsigned at) { return own + at * (4 * T) + 4 * lane; };
    I4Any i = *(const I4Any*)(q + entries(at));
    f4 v = ld_stream(g + entries(at));
    for (unsigned s = 0; s < steps; ++s) {
      at = at + 1 < steps ? at + 1 : 0;
      const I4Any i1 = *(const I4Any*)(q + entries(at));
      const f4 v1 = ld_stream(g + entries(at));
#pragma unroll
      for (int j = 0; j < 4; ++j) i.v[j] = index_of(i.v[j], n);
      take(i, v);
      i = i1;
      v = v1;
    }
  }
  const unsigned e0 = own + steps * (4 * T);
  if (e0 < hi) {
    I4Any i;
    f4 v = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      i.v[j] = -1;   // not an entry
      if (e0 + 4 * lane + j < hi) {
        i.v[j] = index_of(q[e0 + 4 * lane + j], n);
        v[j] = g[e0 + 4 * lane + j];
      }
    }
    take(i, v);
  }
  __syncthreads();
  float* o = grad_points + (long)row * n;
  if (splits == 1)
    for (int k = tid; k < n; k += T) o[k] = (float)srow[k];
  else
    for (int k = tid; k < n; k += T)
      if (srow[k] != 0) unsafeAtomicAdd(o + k, (float)srow[k]);   // (NaN != 0)
}
__global__ __launch_bounds__(NTHREADS) void k_zero(long total, float* __restrict__ q) {
  for (long e = (long)blockIdx.x * NTHREADS + threadIdx.x; e < total; e += (long)gridDim.x * NTHREADS) q[e] = 0.0f;
}
__global__ __launch_bounds__(NTHREADS) void k_group_points_grad(long total, int c, int n, int ms,
                                                                const float* __restrict__ grad_out,
                                                                const int* __restrict__ idx, float* __restrict__ grad_points) {
  const long e = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= total) return;
  const int r = (int)(e % ms);
  const long bc = e / ms;
  const int b = (int)(bc / c);
  const int k = min(max(idx[(long)b * ms + r], 0), n - 1);
  unsafeAtomicAdd(grad_points + bc * n + k, grad_out[e]);
}

// 3 nearest known points of every unknown point: squared distances ascending, ties to the smaller index.
//
// 256 to 8192 known points: every workgroup sorts them (counting sort) into a uniform grid of about two points a cell in
// LDS, 16 bytes a point; a thread visits the 27 cells around its point, rows of neighbouring cells as one range, and then
// whatever else lies within its third distance (which shrinks on the way; rows beyond it are skipped).  The answer is that of
// the pass over all points: distances are evaluated the same way, ordered by (distance, index), and cells are left out only
// if their distance, shortened by far more than the rounding of cell numbers and distances, is above the third one.  Coordinates that
// are not finite (or above 1e18) send the workgroup to the pass over all points.  A workgroup's share of the targets is
// what leaves every CU one workgroup, up to one a thread; the known points stay in registers (R a thread) from the bounds over their
// cells to the sorted list, and their places in the cells are what the counting's additions return.  20000 x 2048 points, 8 samples: 258 us
// looking at all, 47 us with a workgroup to 512 targets (320 of them, two on every fourth CU) that read the points three times, 42 like this, 38 with the
// places of a block's rows read together and a point requested while the one before is looked at.
// More targets than that: two workgroups a CU while their points fit (up to 4063 of them), at 64 registers a lane, and where all of them
// then fit at once the targets are shared by as many as there is room for.  At 70 and 82 registers, one a CU, 16 samples of 20000 x 1000 points
// took 71 us (54 now; 59 with 512 threads a workgroup, three or four a CU, reading the points three times), 16 of 20000 x 3000 77 (60; 79).  Where
// they do not fit at once and four of half the size fit a CU (up to 1519 points), those: a CU then waits for the slowest of eight waves and
// not of sixteen.  12 of 50000 x 1024 86 us with 1024 threads, 79 with 512, 64 of 40000 x 1000 229 and 226; targets outside the known points 197 and 185, 494 and
// 485 (186 and 477 with those that read three times).
constexpr int NN_T = 1024, NN_CELLS = 4096;
struct Nearest3 {
  float d1, d2, d3;
  int i1, i2, i3;
  __device__ __forceinline__ void take(float d, int k) {
    if (d > d3) return;   // (NaN goes on and fails every test below)
    const bool a = d < d1 || (d == d1 && k < i1), m = d < d2 || (d == d2 && k < i2), z = d < d3 || (d == d3 && k < i3);
    if (a) { d3 = d2; i3 = i2; d2 = d1; i2 = i1; d1 = d; i1 = k; }
    else if (m) { d3 = d2; i3 = i2; d2 = d; i2 = k; }
    else if (z) { d3 = d; i3 = k; }
  }
};
template <int T, int R>
__global__ __launch_bounds__(T, R > 4 ? 4 : 8) void k_three_nn_grid(int n, int m, int share, const float* __restrict__ unknown,
                                                        const float* __restrict__ known, float* __restrict__ dist2,
                                                        int* __restrict__ idx) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float4* pts = (float4*)smem_raw;           // [m] x, y, z, index
  int* end = (int*)(pts + m);                // [NN_CELLS + 1]: end[c + 1] = end of cell c's points, end[0] = 0
  __shared__ float red[7][T / 64];
  __shared__ int wsum[T / 64];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float INFV = __builtin_huge_valf();
  const float* kp = known + (long)b * m * 3;
  float lo[3] = {INFV, INFV, INFV}, hi[3] = {-INFV, -INFV, -INFV}, odd = 0.0f;
  float pt[R][3];   // points tid, tid + T, .. (past the end: the last one again, not counted)
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int a = 0; a < 3; ++a) pt[r][a] = kp[min(tid + r * T, m - 1) * 3 + a];
  const int j = blockIdx.x * share + tid;
  const bool live = tid < share && j < n;
  const float* u = unknown + ((long)b * n + min(j, n - 1)) * 3;
  const float ux = u[0], uy = u[1], uz = u[2];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float v = pt[r][a];
      if (!(fabsf(v) < 1e18f)) odd = 1.0f;
      lo[a] = fminf(lo[a], v);
      hi[a] = fmaxf(hi[a], v);
    }
  odd = wave_fmax(odd);
  if (lane == 0) red[6][wave] = odd;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float l = -wave_fmax(-lo[a]), h = wave_fmax(hi[a]);
    if (lane == 0) { red[a][wave] = l; red[3 + a][wave] = h; }
  }
  for (int c = tid; c <= NN_CELLS; c += T) end[c] = 0;
  __syncthreads();
  odd = red[6][0];
#pragma unroll
  for (int a = 0; a < 3; ++a) { lo[a] = red[a][0]; hi[a] = red[3 + a][0]; }
#pragma unroll
  for (int w = 1; w < T / 64; ++w) {
    odd = fmaxf(odd, red[6][w]);
#pragma unroll
    for (int a = 0; a < 3; ++a) { lo[a] = fminf(lo[a], red[a][w]); hi[a] = fmaxf(hi[a], red[3 + a][w]); }
  }
  // cells: cubes of side `side`, at most 32 along an axis and NN_CELLS in all
  const float ext[3] = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
  const float longest = fmaxf(fmaxf(ext[0], ext[1]), ext[2]);
  float side = fmaxf(cbrtf(ext[0] * ext[1] * ext[2] * 2.0f / (float)m), longest * (1.0f / 32.0f));
  if (!(side > 1e-30f)) side = 1.0f;   // all in one place
  int g[3];
  auto count_cells = [&]() {
    for (int a = 0; a < 3; ++a) g[a] = min(max((int)(ext[a] / side) + 1, 1), 33);
    return g[0] * g[1] * g[2];
  };
  while (count_cells() > NN_CELLS) side *= 1.25f;
  const float inv = 1.0f / side;
  auto cell1 = [&](float v, int a) { return min(max((int)((v - lo[a]) * inv), 0), g[a] - 1); };

  Nearest3 best = {INFV, INFV, INFV, 0, 0, 0};
  if (odd == 0.0f && longest < INFV) {   // uniform
    int cell[R], place[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      cell[r] = (cell1(pt[r][2], 2) * g[1] + cell1(pt[r][1], 1)) * g[0] + cell1(pt[r][0], 0);
      if (tid + r * T < m) place[r] = atomicAdd(&end[1 + cell[r]], 1);
    }
    __syncthreads();
    {  // exclusive prefix sum: NN_CELLS / T neighbours per thread
      constexpr int E = NN_CELLS / T;
      int own = 0;
      for (int e = 0; e < E; ++e) own += end[1 + tid * E + e];
      int incl = own;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      if (lane == 63) wsum[wave] = incl;
      __syncthreads();
      int at = incl - own;
      for (int w = 0; w < wave; ++w) at += wsum[w];
      for (int e = 0; e < E; ++e) { at += end[1 + tid * E + e]; end[1 + tid * E + e] = at; }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (tid + r * T < m) pts[end[cell[r]] + place[r]] = make_float4(pt[r][0], pt[r][1], pt[r][2], __builtin_bit_cast(float, tid + r * T));
    __syncthreads();
    if (live) {
      const int cx = cell1(ux, 0), cy = cell1(uy, 1), cz = cell1(uz, 2);
      auto points = [&](int e, int e1) {   // of the sorted list; the next one is on its way while this one is looked at
        if (e >= e1) return;
        float4 p = pts[e];
        for (;;) {
          const float4 next = pts[min(e + 1, m - 1)];
          best.take(sqdist(ux, uy, uz, p.x, p.y, p.z), __builtin_bit_cast(int, p.w));
          if (++e >= e1) break;
          p = next;
        }
      };
      // how near a point of cell row (y, z) can be, squared (0 if it may be nearer than the margin for rounding)
      const float du[3] = {ux - lo[0], uy - lo[1], uz - lo[2]};
      const float margin = 1e-4f * side;
      auto gap = [&](float d, int c) {   // distance along one axis from d to cells' interval number c
        const float q = fmaxf((float)c * side - d, d - (float)(c + 1) * side) * (1.0f - 1e-5f) - margin;
        return q > 0.0f ? q * q : 0.0f;
      };
      // cells x0 .. x1 of row (y, z), unless every point of it is farther than the third one
      auto row = [&](int x0, int x1, int y, int z) {
        const int c = (z * g[1] + y) * g[0];
        if (x0 <= x1 && !(gap(du[1], y) + gap(du[2], z) > best.d3)) points(end[c + x0], end[c + x1 + 1]);
      };
      int a0[3], a1[3];   // the cells visited so far: first the block around the point's own, its row first
      const int cc[3] = {cx, cy, cz};
#pragma unroll
      for (int a = 0; a < 3; ++a) { a0[a] = max(cc[a] - 1, 0); a1[a] = min(cc[a] + 1, g[a] - 1); }
      {
        int from[9], to[9];   // the block's rows, their places read together
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const int y = cy + (t % 3 == 0 ? 0 : t % 3 == 1 ? -1 : 1), z = cz + (t < 3 ? 0 : t < 6 ? -1 : 1);
          const bool in = y >= a0[1] && y <= a1[1] && z >= a0[2] && z <= a1[2];
          const int c = in ? (z * g[1] + y) * g[0] : 0;
          from[t] = end[c + a0[0]];
          to[t] = in ? end[c + a1[0] + 1] : 0;
        }
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const int y = cy + (t % 3 == 0 ? 0 : t % 3 == 1 ? -1 : 1), z = cz + (t < 3 ? 0 : t < 6 ? -1 : 1);
          if (!(gap(du[1], y) + gap(du[2], z) > best.d3)) points(from[t], to[t]);
        }
      }
      for (int r = 2;; r *= 2) {
        // everything within the third distance, if there is one: after that nothing is left to see.  Else a larger block.
        const bool three = best.d3 < INFV;
        const float reach = three ? sqrtf(best.d3) * (1.0f + 1e-5f) + margin : 0.0f;
        int b0[3], b1[3];
        bool same = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          b0[a] = three ? min(max((int)((du[a] - reach) * inv), 0), a0[a]) : max(cc[a] - r, 0);
          b1[a] = three ? max(min((int)fminf((du[a] + reach) * inv, 64.0f), g[a] - 1), a1[a]) : min(cc[a] + r, g[a] - 1);
          same = same && b0[a] == a0[a] && b1[a] == a1[a];
        }
        if (!same)
          for (int z = b0[2]; z <= b1[2]; ++z)
            for (int y = b0[1]; y <= b1[1]; ++y) {
              const bool seen = y >= a0[1] && y <= a1[1] && z >= a0[2] && z <= a1[2];
              row(b0[0], seen ? a0[0] - 1 : b1[0], y, z);
              if (seen) row(a1[0] + 1, b1[0], y, z);
            }
        if (three || (b0[0] == 0 && b0[1] == 0 && b0[2] == 0 && b1[0] == g[0] - 1 && b1[1] == g[1] - 1 && b1[2] == g[2] - 1)) break;
#pragma unroll
        for (int a = 0; a < 3; ++a) { a0[a] = b0[a]; a1[a] = b1[a]; }
      }
    }
  } else if (live) {
    for (int k = 0; k < m; ++k) best.take(sqdist(ux, uy, uz, kp[k * 3], kp[k * 3 + 1], kp[k * 3 + 2]), k);
  }
  if (live) {
    float* dd = dist2 + ((long)b * n + j) * 3;
    int* ii = idx + ((long)b * n + j) * 3;
    dd[0] = best.d1; dd[1] = best.d2; dd[2] = best.d3;
    ii[0] = best.i1; ii[1] = best.i2; ii[2] = best.i3;
  }
}

// Any number of known points.
__global__ __launch_bounds__(NTHREADS) void k_three_nn(int n, int m, const float* __restrict__ unknown,
                                                       const float* __restrict__ known, float* __restrict__ dist2,
                                                       int* __restrict__ idx) {
  __shared__ float kx[NTHREADS], ky[NTHREADS], kz[NTHREADS];
  const int b = blockIdx.y;
  const int j = blockIdx.x * NTHREADS + threadIdx.x;
  const bool live = j < n;
  float ux = 0.0f, uy = 0.0f, uz = 0.0f;
  if (live) {
    const float* u = unknown + ((long)b * n + j) * 3;
    ux = u[0]; uy = u[1]; uz = u[2];
  }
  float b1 = __builtin_huge_valf(), b2 = b1, b3 = b1;  // fewer than 3 known points leave +inf (the reference's 1e40)
  int i1 = 0, i2 = 0, i3 = 0;
  const float* kp = known + (long)b * m * 3;
  for (int k0 = 0; k0 < m; k0 += NTHREADS) {
    const int kk = k0 + threadIdx.x;
    if (kk < m) { kx[threadIdx.x] = kp[kk * 3]; ky[threadIdx.x] = kp[kk * 3 + 1]; kz[threadIdx.x] = kp[kk * 3 + 2]; }
    __syncthreads();
    const int lim = min(NTHREADS, m - k0);
    for (int t = 0; t < lim; ++t) {
      const float d = sqdist(ux, uy, uz, kx[t], ky[t], kz[t]);
      const int k = k0 + t;
      if (d < b1) { b3 = b2; i3 = i2; b2 = b1; i2 = i1; b1 = d; i1 = k; }
      else if (d < b2) { b3 = b2; i3 = i2; b2 = d; i2 = k; }
      else if (d < b3) { b3 = d; i3 = k; }
    }
    __syncthreads();
  }
  if (live) {
    float* dd = dist2 + ((long)b * n + j) * 3;
    int* ii = idx + ((long)b * n + j) * 3;
    dd[0] = b1; dd[1] = b2; dd[2] = b3;
    ii[0] = i1; ii[1] = i2; ii[2] = i3;
  }
}

// out[b][c][j] = sum_k weight[b][j][k] * points[b][c][idx[b][j][k]]
__global__ __launch_bounds__(NTHREADS) void k_three_interpolate(long total, int c, int m, int n, const float* __restrict__ points,
                                                                const int* __restrict__ idx, const float* __restrict__ weight,
                                                                float* __restrict__ out) {
  const long e = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= total) return;
  const int j = (int)(e % n);
  const long bc = e / n;
  const int b = (int)(bc / c);
  const long o = ((long)b * n + j) * 3;
  const float* src = points + bc * m;
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 3; ++k) acc += weight[o + k] * src[min(max(idx[o + k], 0), m - 1)];
  out[e] = acc;
}
__global__ __launch_bounds__(NTHREADS) void k_three_interpolate_grad(long total, int c, int n, int m,
                                                                     const float* __restrict__ grad_out,
                                                                     const int* __restrict__ idx,
                                                                     const float* __restrict__ weight,
                                                                     float* __restrict__ grad_points) {
  const long e = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= total) return;
  const int j = (int)(e % n);
  const long bc = e / n;
  const int b = (int)(bc / c);
  const long o = ((long)b * n + j) * 3;
  float* dst = grad_points + bc * m;
  const float g = grad_out[e];
#pragma unroll
  for (int k = 0; k < 3; ++k) unsafeAtomicAdd(dst + min(max(idx[o + k], 0), m - 1), g * weight[o + k]);
}

// Interpolation with CH channels of the m known points in LDS, [m][CH]: one thread per target and step reads the target's
// indices and weights once for all of them and CH / 4 16-byte LDS reads per neighbour.  Bound by writing the output:
// 256 channels, 2048 -> 20000 points, 8 samples: 166 us with a
// thread per element, 53 us with stores that pass through L2, 45 us here (164 MB written, 3.6 TB/s; under the profiler).
template <int CH>
__global__ __launch_bounds__(512) void k_interp_rows(int c, int m, int n, int splits, unsigned per, const float* __restrict__ points,
                                                     const int* __restrict__ idx, const float* __restrict__ weight,
                                                     float* __restrict__ out) {
  extern __shared__ __align__(16) float srow[];
  const int wg = xcd_remap(blockIdx.x, gridDim.x), per_b = (c + CH - 1) / CH * splits;
  const int tid = threadIdx.x, b = wg / per_b, c0 = (wg % per_b) / splits * CH, part = wg % splits;
  for (int e = tid; e < m * CH; e += 512) {   // neighbouring lanes: neighbouring channels (no bank conflict)
    const int ch = min(c0 + e % CH, c - 1);
    srow[e] = points[((long)b * c + ch) * m + e / CH];
  }
  __syncthreads();
  const unsigned hi = min((part + 1) * per, (unsigned)n);
  for (unsigned j = part * per + tid; j < hi; j += 512) {
    const long o = ((long)b * n + j) * 3;
    f4 acc[CH / 4];
#pragma unroll
    for (int q = 0; q < CH / 4; ++q) acc[q] = (f4){0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float w = weight[o + k];
      const f4* s = (const f4*)(srow + index_of(idx[o + k], m) * CH);
#pragma unroll
      for (int q = 0; q < CH / 4; ++q) {
        const f4 v = s[q];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[q][r] += w * v[r];
      }
    }
#pragma unroll
    for (int ch = 0; ch < CH; ++ch)
      if (c0 + ch < c) __builtin_nontemporal_store(acc[ch / 4][ch % 4], out + ((long)b * c + c0 + ch) * n + j);
  }
}
// Its gradient, all of grad_points (b, c, m) written.  Adding target by target into rows of sums in LDS takes 600 us (8
// samples, 256 channels, 2048 <- 20000 points): an LDS float addition to scattered words runs at a third of a lane a cycle.
// So the targets' three (point, weight) entries are sorted by point first, once for all channels: k_inverse_rank counts and
// gives every entry its place within its point, k_inverse_fill writes the list.  A point's entries fill whole blocks of
// INV_E, so that a lane of k_interp_rows_grad sums a block without asking where a point ends; neighbouring lanes with one
// point add up by row-lane moves, and the last of them writes the sum; what a wave's share of the list has of its first and
// last point meets in LDS.  No atomics: a thread per 59 entries that added every run it finished to the result took 211 us,
// the waits for its list behind those additions in the one counter both have, and one addition at either end of 64 blocks
// still cost 70 of 147 us.  68 us here (164 MB read: 36 at the copy's rate; 52 without reading more than the first rows, 53 with
// one step's part of the list in place of all of it, 78 with row reads that displace the list in L2), 11 + 12 for the list;
// longer blocks or more of the list in flight gave nothing.  397 with atomics into a channel-last buffer.
constexpr int INV_T = 1024, INV_E = 8;
struct InvList {              // per sample `blocks` places
  unsigned* target;           // [place][INV_E / 2] two targets each
  float* weight;              // [INV_E / 4][place][4]
  unsigned* point;            // entries << 16 | point
  int *count, *first, *rank;  // [m] entries of a point, [m + 1] its first block (last: all blocks), [3 n] places in the point
  int blocks;
  // most blocks that 3 n entries of m points can take
  static long most(long n, long m) { return (3 * n + (INV_E - 1) * std::min(3 * n, m)) / INV_E + 1; }
  static long ints(long b, long n, long m) { return b * (most(n, m) * (INV_E / 2 + INV_E + 1) + 2 * m + 1 + 3 * n); }
  InvList(int* ws, long b, long n, long m) : blocks((int)most(n, m)) {
    target = (unsigned*)ws;
    weight = (float*)(target + b * blocks * (INV_E / 2));
    point = (unsigned*)(weight + b * blocks * INV_E);
    count = (int*)(point + b * blocks);
    first = count + b * m;
    rank = first + b * (m + 1);
  }
};
__global__ __launch_bounds__(INV_T) void k_inverse_rank(int n, int m, const int* __restrict__ idx, InvList l) {
  extern __shared__ int cnt[];
  __shared__ int wsum[INV_T / 64];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int k = tid; k < m; k += INV_T) cnt[k] = 0;
  __syncthreads();
  const int* q = idx + (long)b * n * 3;
  int* r = l.rank + (long)b * n * 3;
  constexpr int U = 16;   // entries of a thread in flight: one workgroup a sample, so latency is all there is (20 us with four)
  for (int e0 = tid; e0 < 3 * n; e0 += INV_T * U) {
    int k[U];
#pragma unroll
    for (int u = 0; u < U; ++u) k[u] = index_of(q[min(e0 + INV_T * u, 3 * n - 1)], m);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + INV_T * u < 3 * n) k[u] = atomicAdd(cnt + k[u], 1);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + INV_T * u < 3 * n) r[e0 + INV_T * u] = k[u];
  }
  __syncthreads();
  const int per = (m + INV_T - 1) / INV_T, k0 = tid * per, k1 = min(k0 + per, m);
  int own = 0;
  for (int k = k0; k < k1; ++k) own += (cnt[k] + INV_E - 1) / INV_E;
  int incl = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int at = incl - own;
  for (int w = 0; w < wave; ++w) at += wsum[w];
  int* first = l.first + (long)b * (m + 1);
  for (int k = k0; k < k1; ++k) {
    first[k] = at;
    l.count[(long)b * m + k] = cnt[k];
    at += (cnt[k] + INV_E - 1) / INV_E;
  }
  if (tid == INV_T - 1) first[m] = at;
}
// Writes the list and clears the result (the sums of points that two waves meet at are added to it).
__global__ __launch_bounds__(NTHREADS) void k_inverse_fill(int n, int m, const int* __restrict__ idx, const float* __restrict__ weight,
                                                           InvList l, int pad, long total, float* __restrict__ grad_points) {
  const int b = blockIdx.y, e = blockIdx.x * NTHREADS + threadIdx.x;
  const long threads = (long)gridDim.x * gridDim.y * NTHREADS;
  for (long z = ((long)b * gridDim.x + blockIdx.x) * NTHREADS + threadIdx.x; z < total; z += threads) grad_points[z] = 0.0f;
  if (e >= 3 * n) return;
  const int k = index_of(idx[(long)b * n * 3 + e], m), r = l.rank[(long)b * n * 3 + e], cnt = l.count[(long)b * m + k];
  const long base = (long)b * l.blocks, at = base + l.first[(long)b * (m + 1) + k] + r / INV_E;
  unsigned short* t = (unsigned short*)(l.target + at * (INV_E / 2));
  auto put = [&](int i, int target, float w) {
    t[i] = (unsigned short)target;
    l.weight[((base * (INV_E / 4)) + (long)(i / 4) * l.blocks + (at - base)) * 4 + i % 4] = w;
  };
  put(r % INV_E, e / 3, weight[(long)b * n * 3 + e]);
  if (r % INV_E == 0) l.point[at] = (unsigned)min(cnt - r, INV_E) << 16 | (unsigned)k;
  if (r == cnt - 1)
    for (int i = r % INV_E + 1; i < INV_E; ++i) put(i, pad, 0.0f);
}
constexpr unsigned NO_POINT = 0xffffu;
static_assert(ROW_POINTS < (int)NO_POINT, "no point has this number, and a target fits in 16 bits");
// R rows of grad_out in LDS, a target's R values side by side, and behind them the value zero that the entries filling up a
// block read (a weight of zero alone would not do: zero times a gradient that is no number is none); where the row itself
// takes all of the LDS (ZERO = false) such entries are told by the block's count.
// PIPE: a workgroup takes `per` of the `sets` of R rows one after the other and asks for the next one's while it sums.  The rows
// fill the CU's LDS, so no other workgroup's requests are in flight meanwhile, and reading and summing added up.  They are asked for
// a piece a step, each behind the step's part of the list: what a wave asks for arrives in order, and the list is not to wait for
// rows that are not needed yet.  8 samples, 256 channels, 2048 <- 20000
// points: 84 -> 82 us so, 69 with the rows put into LDS 16 bytes at a time and read from there 8, 68 with fewer instructions.
template <int R, bool ZERO, bool PIPE>
__global__ __launch_bounds__(INV_T, PIPE ? 4 : 8) void k_interp_rows_grad(int c, int n, int m, const float* __restrict__ grad_out, InvList l,
                                                           float* __restrict__ grad_points, int sets, int per) {
  extern __shared__ __align__(16) float lds[];
  float* srow = (float*)__builtin_assume_aligned(lds, 16);   // (the declaration's alignment alone gives accesses of two single words)
  typedef float Vals __attribute__((ext_vector_type(R)));
  typedef unsigned u4_any __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int T = INV_T;
  const int wg = xcd_remap(blockIdx.x, gridDim.x), per_b = (c + R - 1) / R;   // an XCD's workgroups: one sample's list in its L2
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // sums of a point over the lanes before (a point's lanes lie side by side); on: one point from the row's first lane, or from
  // as far back as the step looks, to here
  auto scan = [&](unsigned k, float (&s)[R]) {
    const bool begins = __builtin_amdgcn_update_dpp(-1, (int)k, 0x138, 0xf, 0xf, false) != (int)k || lane == 0;
    const int back = __builtin_clzll(__ballot(begins) << (63 - lane));   // lanes before it with its point
    // a lane whose run reaches back `far` lanes or more takes what `ctrl` moves to it (by mask: zero times no number is none)
    auto step = [&](auto ctrl, int far) {
      int on = (far - 1 - back) >> 31;
      asm("" : "+v"(on));
#pragma unroll
      for (int r = 0; r < R; ++r)
        s[r] += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s[r]), decltype(ctrl)::value, 0xf, 0xf, true) & on);
    };
    step(std::integral_constant<int, 0x111>{}, 1);   // from one, two, four, eight lanes before, inside a row of 16
    step(std::integral_constant<int, 0x112>{}, 2);
    step(std::integral_constant<int, 0x114>{}, 4);
    step(std::integral_constant<int, 0x118>{}, 8);
    step(std::integral_constant<int, 0x142>{}, lane & 16 ? (lane & 15) + 1 : 64);   // from the last lane of the row before
    step(std::integral_constant<int, 0x143>{}, lane & 32 ? lane - 31 : 64);         // from lane 31
  };
  auto after = [&](unsigned k) {   // the next lane's
    return (unsigned)__builtin_amdgcn_update_dpp(-1, (int)k, 0x130, 0xf, 0xf, false);
  };
  // a set's rows in registers, a piece of 4 T of each at a time: U pieces, then the rows' last elements
  constexpr int PIECES = (ROW_POINTS / R + 4 * T - 1) / (4 * T), U = PIPE ? PIECES : R == 1 ? 5 : R == 2 ? 2 : 1;
  // (not PIPE: two workgroups of 16 waves a CU, so 64 registers.  Two pieces of four rows took 66, and were one too many for the rows
  // of up to 4095 that all are in one; 8 samples, 256 channels, 512 <- 3000 points 14.8 -> 11.7 us, 1024 <- 5000 20.3 -> 17.5; 16 samples,
  // 256 <- 1024 17.4 -> 12.7)
  f4 v[U][R];
  float vt[R];
  // piece `at` of set q into v[u]; where there is none, or with n < 4, anything that can be read
  auto ask = [&](int u, int q, int at, bool real) {
    const int c0 = (q % per_b) * R;
    const float* row = real ? grad_out + ((long)(q / per_b) * c + c0) * n : l.weight;
    const int k = real ? min(4 * (tid + T * at), n - 4) : 0, hop = real ? n : 0;
#pragma unroll
    for (int r = 0; r < R; ++r) v[u][r] = ld_stream(row + (long)min(r, c - c0 - 1) * hop + k);
  };
  auto ask_tail = [&](int q) {
    const int c0 = (q % per_b) * R;
    const float* row = grad_out + ((long)(q / per_b) * c + c0) * n;
#pragma unroll
    for (int r = 0; r < R; ++r) vt[r] = row[(long)min(r, c - c0 - 1) * n + min((n & ~3) + tid, n - 1)];
  };
  auto keep = [&](int u, int at) {
    const int k = 4 * (tid + T * at);
    if (k + 3 < n) {
#pragma unroll
      for (int i = 0; i < R; ++i) {   // 16 bytes at a time: lane addresses are 16 R apart, and narrower accesses met in as many banks
        f4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = v[u][(4 * i + e) % R][(4 * i + e) / R];
        *(f4*)(srow + k * R + 4 * i) = w;
      }
    }
  };
  if (n == 0) return;
  const int set0 = PIPE ? wg * per : wg, set1 = PIPE ? min(set0 + per, sets) : wg + 1;
  if (PIPE && set0 < set1) {
#pragma unroll
    for (int u = 0; u < U; ++u) ask(u, set0, u, n >= 4);
    ask_tail(set0);
  }
  for (int set = set0; set < set1; ++set) {
    const int b = set / per_b, c0 = (set % per_b) * R, nch = min(R, c - c0);
    const int blocks = l.first[(long)b * (m + 1) + m];
    const long base = (long)b * l.blocks;
    const unsigned* pt = l.point + base;
    const u4_any* tg = (const u4_any*)(l.target + base * (INV_E / 2));
    const f4_stream *w0 = (const f4_stream*)(l.weight + base * INV_E), *w1 = w0 + l.blocks;
    float* o = grad_points + ((long)b * c + c0) * m;
    auto put = [&](unsigned k, const float (&s)[R]) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r < nch) *(float*)((char*)(o + (long)r * m) + 4 * k) = s[r];
    };
    // a wave's share of the list, 64 blocks a step.  first: the share's first point, to which earlier waves may have something
    // to add, and its sum (head) once it has ended; open, carry: the point of the step's last block and its sum so far
    const int share = (blocks + T / 64 - 1) / (T / 64), end = min(blocks, (wave + 1) * share);
    int at = wave * share;   // uniform
    struct Block { unsigned p; u4_any t; f4 wa, wb; };
    auto load = [&](int at) {
      const unsigned i = min(at + lane, blocks - 1), i4 = i * 4, i16 = i * 16;   // (a list has less than 2^26 places)
      return Block{*(const unsigned*)((const char*)pt + i4), *(const u4_any*)((const char*)tg + i16),
                   *(const f4_stream*)((const char*)w0 + i16), *(const f4_stream*)((const char*)w1 + i16)};
    };
    Block q0 = load(at);
    if constexpr (PIPE) {
#pragma unroll
      for (int u = 0; u < U; ++u) keep(u, u);
    } else {
      for (int p0 = 0; 4 * T * p0 + 3 < n; p0 += U) {   // uniform
#pragma unroll
        for (int u = 0; u < U; ++u) ask(u, set, p0 + u, true);
#pragma unroll
        for (int u = 0; u < U; ++u) keep(u, p0 + u);
      }
      ask_tail(set);
    }
    if ((n & ~3) + tid < n)
#pragma unroll
      for (int r = 0; r < R; ++r) srow[((n & ~3) + tid) * R + r] = vt[r];
    if (ZERO && tid < R) srow[n * R + tid] = 0.0f;
    __syncthreads();
    unsigned open = NO_POINT;
    bool ended = false;
    float carry[R], head[R];
#pragma unroll
    for (int r = 0; r < R; ++r) carry[r] = head[r] = 0.0f;
    const unsigned first = __builtin_amdgcn_readfirstlane(q0.p & 0xffffu);
    auto take = [&](const Block& q, int at) {
      const unsigned k = at + lane < end ? q.p & 0xffffu : NO_POINT;
      float s[R];
#pragma unroll
      for (int r = 0; r < R; ++r) s[r] = 0.0f;
#pragma unroll
      for (int e = 0; e < INV_E; ++e) {
        unsigned j = e & 1 ? q.t[e / 2] >> 16 : q.t[e / 2] & 0xffffu;
        asm("" : "+v"(j));   // (else the masking moves behind the scaling and takes an instruction more)
        const Vals x = *(const Vals*)(srow + j * R);
        const float w = e < 4 ? q.wa[e & 3] : q.wb[e & 3];
#pragma unroll
        for (int r = 0; r < R; ++r) s[r] += w * (ZERO || e < (int)(q.p >> 16) ? x[r] : 0.0f);
      }
      scan(k, s);
      const int last = min(63, end - 1 - at);   // of the step's blocks
      const unsigned k0 = (unsigned)__builtin_amdgcn_readlane((int)k, 0), k_last = (unsigned)__builtin_amdgcn_readlane((int)k, last);
      if (k0 == open) {
#pragma unroll
        for (int r = 0; r < R; ++r) s[r] += k == k0 ? carry[r] : 0.0f;
      } else if (open != NO_POINT) {   // it ended with the last step
        if (open == first) {
          ended = true;
#pragma unroll
          for (int r = 0; r < R; ++r) head[r] = carry[r];
        } else if (lane == 0) put(open, carry);
      }
      if (k0 == first && k_last != first) {
        ended = true;
        const int l = __popcll(__ballot(k == first)) - 1;
#pragma unroll
        for (int r = 0; r < R; ++r) head[r] = lane_f(s[r], l);
      }
      if (lane < last && after(k) != k && k != first) put(k, s);
      open = k_last;
#pragma unroll
      for (int r = 0; r < R; ++r) carry[r] = lane_f(s[r], last);
    };
    if constexpr (PIPE) {
      const int next = min(set + 1, set1 - 1);
      const bool real = set + 1 < set1 && n >= 4;
      for_each_slot<U>([&](auto piece) {
        const Block n0 = load(at + 64);
        ask(decltype(piece)::value, next, decltype(piece)::value, real);
        if (at < end) take(q0, at);   // uniform
        q0 = n0;
        at += 64;
      });
      ask_tail(next);
    }
    for (; at < end; at += 64) {   // uniform
      const Block n0 = load(at + 64);
      take(q0, at);
      q0 = n0;
    }
    // the waves' first and last points, in order
    __syncthreads();
    if (lane < 2) {
      float* e = srow + (wave * 2 + lane) * (R + 1);
      e[0] = __builtin_bit_cast(float, lane == 0 && ended ? first : open);
#pragma unroll
      for (int r = 0; r < R; ++r) e[1 + r] = lane ? carry[r] : ended ? head[r] : 0.0f;
    }
    __syncthreads();
    if (tid < 64) {
      const bool in = lane < T / 32;
      const float* e = srow + (in ? lane : 0) * (R + 1);
      const unsigned k = in ? __builtin_bit_cast(unsigned, e[0]) : NO_POINT;
      float s[R];
#pragma unroll
      for (int r = 0; r < R; ++r) s[r] = e[1 + r];
      scan(k, s);
      if (after(k) != k && k != NO_POINT) put(k, s);
    }
    if (PIPE) __syncthreads();   // the next set's rows take the place of these sums
  }
}

// Gradients into a channel-last buffer, out_cl (b, n, c) += ...: a 64 x 64 tile of grad_out (channels x entries) is
// read along the entries (coalesced), turned in LDS, and added with lanes running over channels, so one atomic
// instruction covers 64 consecutive floats of one point instead of 64 scattered cache lines.
// K3 == false: grouping, entries e = (j, s) with index idx[b][e], value grad_out[b][ch][e];
// K3 == true: interpolation, entries j with three indices and weights each, value grad_out[b][ch][j] * weight[b][j][k].
template <bool K3>
__global__ __launch_bounds__(NTHREADS) void k_scatter_channel_last(int c, int n, int ne, const float* __restrict__ grad_out,
                                                                   const int* __restrict__ idx, const float* __restrict__ weight,
                                                                   float* __restrict__ out_cl) {
  __shared__ float tile[64][65];
  const int b = blockIdx.z, c0 = blockIdx.y * 64, e0 = blockIdx.x * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int r = wave; r < 64; r += NTHREADS / 64) {
    const int ch = c0 + r, e = e0 + lane;
    tile[r][lane] = (ch < c && e < ne) ? grad_out[((long)b * c + ch) * ne + e] : 0.0f;
  }
  __syncthreads();
  const int ch = c0 + lane;
  for (int r = wave; r < 64; r += NTHREADS / 64) {
    const int e = e0 + r;
    if (e >= ne) break;  // wave-uniform
    const float g = tile[lane][r];
    if (K3) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const long o = ((long)b * ne + e) * 3 + k;
        const int p = min(max(idx[o], 0), n - 1);
        if (ch < c) unsafeAtomicAdd(out_cl + ((long)b * n + p) * c + ch, g * weight[o]);
      }
    } else {
      const int p = min(max(idx[(long)b * ne + e], 0), n - 1);
      if (ch < c) unsafeAtomicAdd(out_cl + ((long)b * n + p) * c + ch, g);
    }
  }
}

int launch_scatter_channel_last(bool k3, int b, int c, int n, int ne, const float* grad_out, const int* idx,
                                const float* weight, float* out_cl, hipStream_t st) {
  const dim3 g((ne + 63) / 64, (c + 63) / 64, b), t(NTHREADS);
  if (k3) hipLaunchKernelGGL(k_scatter_channel_last<true>, g, t, 0, st, c, n, ne, grad_out, idx, weight, out_cl);
  else hipLaunchKernelGGL(k_scatter_channel_last<false>, g, t, 0, st, c, n, ne, grad_out, idx, weight, out_cl);
  return (int)hipGetLastError();
}

static unsigned blocks_for(long total) { return (unsigned)((total + NTHREADS - 1) / NTHREADS); }
static unsigned zero_blocks(long total) { return (unsigned)std::min<long>(blocks_for(std::min(total, 1L << 31)), 1 << 20); }

int launch_fps(int b, int n, int npoint, const float* xyz, float* temp, int* idxs, hipStream_t st) {
#define FPS_GROUPS(W, S) hipLaunchKernelGGL((k_fps_groups<W, S>), dim3(b), dim3(64 * W), 0, st, n, npoint, xyz, idxs)
  // Eight waves up to 2048 points (fewer meet at the barrier: 0.565 against 0.58 us a draw at 2048), sixteen above (0.590
  // against 0.593 at 4096, 0.65 against 0.67 at 8192, 0.76 against 0.94 at 20000); slots just enough for n.
  if (n <= 64 * 8 * 4) FPS_GROUPS(8, 4);
  else if (n <= 64 * 16 * 4) FPS_GROUPS(16, 4);
  else if (n <= 64 * 16 * 8) FPS_GROUPS(16, 8);
  else if (n <= 64 * 16 * 12) FPS_GROUPS(16, 12);
  else if (n <= 64 * 16 * 16) FPS_GROUPS(16, 16);
  else if (n <= 64 * 16 * 20) FPS_GROUPS(16, 20);
  else if (n <= 64 * 16 * 24) FPS_GROUPS(16, 24);
  else hipLaunchKernelGGL(k_fps, dim3(b), dim3(FPS_T), 0, st, n, npoint, xyz, temp, idxs);
#undef FPS_GROUPS
  return (int)hipGetLastError();
}
int launch_ball_query(int b, int n, int m, float radius, int nsample, const float* new_xyz, const float* xyz, int* idx,
                      hipStream_t st) {
  // four centres a wave where that leaves a workgroup for every CU
  if ((long)b * ((m + 63) / 64) >= 256)
    hipLaunchKernelGGL(k_ball_query<4>, dim3((m + 63) / 64, b), dim3(BQ_T), 0, st, n, m, radius, radius * radius, nsample, new_xyz, xyz, idx);
  else
    hipLaunchKernelGGL(k_ball_query<1>, dim3((m + 15) / 16, b), dim3(BQ_T), 0, st, n, m, radius, radius * radius, nsample, new_xyz, xyz, idx);
  return (int)hipGetLastError();
}
template <typename K>
static int set_lds_rows(K kern, size_t bytes) {
  return bytes > 64 * 1024 ? (int)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) : 0;
}
// How the entries of a row are cut: about two workgroups per CU in all, but no part shorter than what it costs to put the
// row into LDS (or to clear it and write it back), and a multiple of `unit` entries each.
static int parts_of(long row_blocks, long entries, int row_len, int unit, unsigned* per) {
  long parts = (512 + row_blocks - 1) / row_blocks;
  parts = std::max<long>(1, std::min<long>(parts, entries / std::max(row_len, 2048)));
  *per = (unsigned)(((entries + parts - 1) / parts + unit - 1) / unit * unit);
  return (int)((entries + *per - 1) / *per);
}
static int row_threads(int n) { return n > 10240 ? 1024 : 512; }   // above, at most three workgroups fit a CU's LDS

int launch_group_points(int b, int c, int n, int npoints, int nsample, const float* xyz, const float* centre, float scale,
                        const float* points, const int* idx, float* out, hipStream_t st) {
  GroupP g;
  g.c = c; g.cx = xyz ? 3 : 0; g.n = n; g.ms = npoints * nsample; g.npoints = npoints; g.nsample = nsample;
  g.xyz = xyz; g.centre = centre; g.points = points; g.idx = idx; g.out = out; g.scale = scale;
  const long rows = (long)b * (g.cx + c);
  if (rows > 0x7fffffff) return (int)hipErrorInvalidValue;
  g.rows = (int)rows;
  // rows in LDS where one fits and has at least as many entries as it has points to read, and there are rows for the chip
  if (n <= ROW_POINTS && g.ms >= n) {
    const long total = rows * g.ms, places = 256L * std::max(1, std::min(4, ROW_POINTS / n));
    const long shares = std::max<long>(1, std::min<long>(places, total / std::max(n, 4096)));
    g.share = (total + shares - 1) / shares;
    if (int e = set_lds_rows(&k_group_rows, n * sizeof(float))) return e;
    hipLaunchKernelGGL(k_group_rows, dim3((unsigned)((total + g.share - 1) / g.share)), dim3(row_threads(n)), n * sizeof(float), st, g);
  } else {
    hipLaunchKernelGGL(k_group_points, dim3(blocks_for(g.ms), (unsigned)std::min<long>(rows, 65535)),
                       dim3(NTHREADS), 0, st, g);
  }
  return (int)hipGetLastError();
}
int launch_group_rows_grad(int b, int c, int c0, int cdim, int n, int ms, const float* grad_out, const int* idx,
                           float* grad_points, hipStream_t st) {
  const long rows = (long)b * c;
  unsigned per;
  const int splits = parts_of(rows, ms, n, 256, &per);
  if (splits > 1) hipLaunchKernelGGL(k_zero, dim3(zero_blocks(rows * n)), dim3(NTHREADS), 0, st, rows * n, grad_points);
  auto go = [&](auto kern, size_t bytes, int threads) -> int {
    if (int e = set_lds_rows(kern, bytes)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)(rows * splits)), dim3(threads), bytes, st, c, c0, cdim, n, ms, splits, per, grad_out, idx,
                       grad_points);
    return 0;
  };
  const int e = n <= WIDE_POINTS ? go(&k_group_rows_grad<true>, n * sizeof(double), 512)
                                 : go(&k_group_rows_grad<false>, n * sizeof(float), row_threads(n));
  if (e) return e;
  return (int)hipGetLastError();
}
int launch_group_points_grad(int b, int c, int n, int ms, const float* grad_out, const int* idx, float* grad_points,
                             hipStream_t st) {
  const long total = (long)b * c * ms;
  hipLaunchKernelGGL(k_group_points_grad, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, n, ms, grad_out, idx,
                     grad_points);
  return (int)hipGetLastError();
}
int launch_three_nn(int b, int n, int m, const float* unknown, const float* known, float* dist2, int* idx, hipStream_t st) {
  if (m >= 256 && m <= 8192) {   // fewer: building the grid costs as much as looking at all; more: they do not fit in LDS
    const size_t sm = m * sizeof(float4) + (NN_CELLS + 1) * sizeof(int);
    const int room = 2 * (sm + 512) <= 160 * 1024 ? 2 * NCU : NCU;   // workgroups at once; 512: the kernel's own LDS
    int groups = std::max((n + NN_T - 1) / NN_T, std::min(std::max(NCU / b, 1), (n + 127) / 128));
    if ((long)groups * b > NCU && (long)groups * b <= room) groups = room / b;
    const bool halves = (long)groups * b > 2 * NCU && m <= 3 * NN_T / 2 && 4 * (sm + 256) <= 160 * 1024;
    const int share = halves ? NN_T / 2 : (n + groups - 1) / groups;
    auto go = [&](auto kern, int threads = NN_T) -> int {
      if (int e = set_lds_rows(kern, sm)) return e;
      hipLaunchKernelGGL(kern, dim3((n + share - 1) / share, b), dim3(threads), sm, st, n, m, share, unknown, known, dist2, idx);
      return 0;
    };
    if (int e = halves ? go(&k_three_nn_grid<NN_T / 2, 3>, NN_T / 2) : m <= 2 * NN_T ? go(&k_three_nn_grid<NN_T, 2>)
                : m <= 4 * NN_T ? go(&k_three_nn_grid<NN_T, 4>) : go(&k_three_nn_grid<NN_T, 8>)) return e;
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(k_three_nn, dim3((n + NTHREADS - 1) / NTHREADS, b), dim3(NTHREADS), 0, st, n, m, unknown, known, dist2,
                     idx);
  return (int)hipGetLastError();
}
int launch_three_interpolate(int b, int c, int m, int n, const float* points, const int* idx, const float* weight, float* out,
                             hipStream_t st) {
  const long total = (long)b * c * n;
  // rows in LDS, see launch_group_points; below two million elements filling LDS takes longer than it saves (64 channels,
  // 400 -> 3000 points, 2 samples: 12 us against 4)
  if (n >= m && total >= 1 << 21 && m <= INTERP_POINTS) {
    const int ch = m <= INTERP_POINTS / 4 ? 8 : 4, groups = (c + ch - 1) / ch;
    const size_t sm = (size_t)m * ch * sizeof(float);
    unsigned per;
    const int splits = parts_of((long)b * groups, n, m, 512, &per);
    if (ch == 8) {
      if (int e = set_lds_rows(&k_interp_rows<8>, sm)) return e;
      hipLaunchKernelGGL(k_interp_rows<8>, dim3(groups * splits * b), dim3(512), sm, st, c, m, n, splits, per, points, idx, weight, out);
    } else {
      if (int e = set_lds_rows(&k_interp_rows<4>, sm)) return e;
      hipLaunchKernelGGL(k_interp_rows<4>, dim3(groups * splits * b), dim3(512), sm, st, c, m, n, splits, per, points, idx, weight, out);
    }
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(k_three_interpolate, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, m, n, points, idx, weight,
                     out);
  return (int)hipGetLastError();
}
long interp_rows_grad_ints(int b, int n, int m) { return InvList::ints(b, n, m); }
int launch_interp_rows_grad(int b, int c, int n, int m, const float* grad_out, const int* idx, const float* weight, int* ws,
                            float* grad_points, hipStream_t st) {
  const InvList l(ws, b, n, m);
  const long total = (long)b * c * m;
  const int zero = n < ROW_POINTS ? 1 : 0;
  if (int e = set_lds_rows(&k_inverse_rank, m * sizeof(int))) return e;
  hipLaunchKernelGGL(k_inverse_rank, dim3(b), dim3(INV_T), m * sizeof(int), st, n, m, idx, l);
  hipLaunchKernelGGL(k_inverse_fill, dim3(blocks_for(std::max(3L * n, 1L)), b), dim3(NTHREADS), 0, st, n, m, idx, weight, l, zero ? n : 0, total, grad_points);
  const auto lds = [&](int r) { return std::max((size_t)r * (n + zero), (size_t)INV_T / 32 * (r + 1)) * sizeof(float); };
  // Sets of rows one after the other in a workgroup (PIPE): where one workgroup's rows leave no room on a CU for a second and there
  // is more than one set for each CU.
  auto go = [&](auto kern, auto pipe, int r) -> int {
    const int sets = (c + r - 1) / r * b;
    const bool one = lds(r) > 80 * 1024 && sets > 256;
    const int per = one ? (sets + 255) / 256 : 1;
    auto launch = [&](auto k) -> int {
      if (int e = set_lds_rows(k, lds(r))) return e;
      hipLaunchKernelGGL(k, dim3((sets + per - 1) / per), dim3(INV_T), lds(r), st, c, n, m, grad_out, l, grad_points, sets, per);
      return 0;
    };
    return one ? launch(pipe) : launch(kern);
  };
  int e;
  if (n < ROW_POINTS / 4 && (long)b * ((c + 3) / 4) >= 256) e = go(&k_interp_rows_grad<4, true, false>, &k_interp_rows_grad<4, true, true>, 4);
  else if (n < ROW_POINTS / 2 && (long)b * ((c + 1) / 2) >= 256) e = go(&k_interp_rows_grad<2, true, false>, &k_interp_rows_grad<2, true, true>, 2);
  else e = zero ? go(&k_interp_rows_grad<1, true, false>, &k_interp_rows_grad<1, true, true>, 1) : go(&k_interp_rows_grad<1, false, false>, &k_interp_rows_grad<1, false, true>, 1);
  return e ? e : (int)hipGetLastError();
}
int launch_three_interpolate_grad(int b, int c, int n, int m, const float* grad_out, const int* idx, const float* weight,
                                  float* grad_points, hipStream_t st) {
  const long total = (long)b * c * n;
  hipLaunchKernelGGL(k_three_interpolate_grad, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, n, m, grad_out, idx,
                     weight, grad_points);
  return (int)hipGetLastError();
}

}  // namespace issm
