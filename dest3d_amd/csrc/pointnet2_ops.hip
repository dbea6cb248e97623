// Point-set operators of the PointNet++ backbone for gfx950: furthest point sampling, ball query, grouping,
// gathering, 3-nearest-neighbour search and interpolation (the functions of the reference's `pointnet2._ext`,
// pointnet2/_ext_src/src/*.cpp).  Index arithmetic is exact; all tensors fp32 / int32, contiguous.
//
//  * furthest point sampling: one workgroup per sample; up to 24576 points live in registers with their running minimum
//    distance, sorted into groups of 64 neighbours so that a draw looks only at groups it can change; beyond that
//    coordinates are re-read and distances kept in the caller's `temp`.  Ties go to the smaller index.
//  * ball query: one wave per query centre; 64 points are tested per step and compacted in index order with a
//    ballot, so the first `nsample` hits are found without a serial scan; the wave stops as soon as it has them.
//  * 3-NN: one thread per unknown point, known points staged through LDS 256 at a time.
//  * group / gather / interpolate: one thread per output element, innermost index fastest; the gradients scatter
//    with hardware float atomics (duplicates in idx are the rule), as the reference does -- either straight into
//    the (b, c, n) layout, one scattered cache line per lane, or (the *_cl entry points) into a channel-last
//    (b, n, c) buffer through an LDS transpose, 64 consecutive floats per instruction.
#include <type_traits>

#include "issm_dev.h"

namespace issm {

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
// of the lanes in `cand`, the one with the smallest `key` (rare: equal distances)
__device__ __forceinline__ int lane_of_least(unsigned long long cand, int key) {
  int best = __builtin_ctzll(cand), bk = __builtin_amdgcn_readlane(key, best);
  for (cand &= cand - 1; cand; cand &= cand - 1) {
    const int l = __builtin_ctzll(cand), k = __builtin_amdgcn_readlane(key, l);
    if (k < bk) { bk = k; best = l; }
  }
  return best;
}

// Up to 64 W S points: one workgroup of W waves per sample, points in registers, and only those looked at that a draw can
// change.  The draws are a serial chain, so what counts is the time of one: passing over all points costs 40 distances
// per lane at 20000 points (1.92 us a draw, the vector unit of one CU saturated).  Here the points are first sorted along a
// Z-order curve over a 16^3 grid (counting sort in LDS) and cut into groups of 64 neighbours, one point per lane; group g
// belongs to wave g % W (neighbouring groups to different waves) as its slot g / W, and lane l of the wave keeps slot l's
// bounding box, largest running distance and the point that has it.  A draw at o compares o's distance to every box with
// the group's largest distance -- one instruction sequence for all groups of a wave -- and goes through the points of
// those groups only that are nearer: about 10 of 313.  One barrier per draw (the waves' bests go through LDS buffers used
// in turn).  20000 points, 2048 draws, 8 samples: 3.93 ms -> 1.97 ms (0.96 us a
// draw: a chain of about 100 dependent instructions, two LDS round trips and a barrier).
//
// The pruning is exact: fp32 rounding is monotone, so for a point q of the box each step of the box's squared distance
// (subtract, square, add, in sqdist's order) is at most the same step for q, and where the box's distance is not below the
// group's largest running distance, no minimum of the group changes.  A NaN anywhere makes the comparison fail, which means
// "look".  Equal distances go to the smaller index at every level, as a pass over all points in order would decide.
constexpr int FPS_CELLS = 4096;   // 16^3
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
  __shared__ int hist[FPS_CELLS];
  __shared__ unsigned short order[T * S];
  __shared__ float red[6][W];
  __shared__ int wsum[W];
  struct alignas(16) Best { unsigned d; float x, y, z; };
  __shared__ Best best[2][W];
  __shared__ int best_pos[2][W];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* p = xyz + (long)b * n * 3;
  int* out = idxs + (long)b * npoint;
  const float INFV = __builtin_huge_valf();

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
  for (int c = tid; c < FPS_CELLS; c += T) hist[c] = 0;
  __syncthreads();
  float ext = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    for (int w = 0; w < W; ++w) { lo[a] = fminf(w ? lo[a] : INFV, red[a][w]); hi[a] = fmaxf(w ? hi[a] : -INFV, red[3 + a][w]); }
    ext = fmaxf(ext, hi[a] - lo[a]);
  }
  const float inv = ext > 0.0f && ext < INFV ? 16.0f / ext : 0.0f;
  auto cell = [&](int k) {
    unsigned c = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      c |= spread4((unsigned)imin(imax((int)((p[k * 3 + a] - lo[a]) * inv), 0), 15)) << a;
    return c;
  };
  for (int k = tid; k < n; k += T) atomicAdd(&hist[cell(k)], 1);
  __syncthreads();
  {  // exclusive prefix sum of the histogram: FPS_CELLS / T neighbours per thread
    constexpr int E = FPS_CELLS / T;
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
    const bool any = __ballot(in) != 0;
    if (lane == j) {
      blx = lx; bly = ly; blz = lz; bhx = hx; bhy = hy; bhz = hz;
      gd = any ? far : 0u;
    }
  });
  float ox = p[0], oy = p[1], oz = p[2];
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
        d[j] = umin(d[j], __builtin_bit_cast(unsigned, sqdist(px[j], py[j], pz[j], ox, oy, oz)) + 1u);
        const unsigned m = wave_max<4>(d[j]);
        const unsigned long long cand = __ballot(d[j] == m);
        const int base = (j * W + wave) * 64;
        int l = __builtin_ctzll(cand);
        if (cand & (cand - 1)) l = lane_of_least(cand, base + lane < n ? (int)order[base + lane] : 0x7fffffff);
        const float x = lane_f(px[j], l), y = lane_f(py[j], l), z = lane_f(pz[j], l);
        if (lane == j) { gd = m; gpos = base + l; gx = x; gy = y; gz = z; }
      });
    });
    // the wave's best, then the workgroup's
    {
      const unsigned m = wave_max<(S > 16 ? 2 : 1)>(gd);
      const unsigned long long cand = __ballot(gd == m);
      int l = __builtin_ctzll(cand);
      if (m && (cand & (cand - 1))) l = lane_of_least(cand, (int)order[gpos]);
      if (lane == l) { best[s & 1][wave] = Best{gd, gx, gy, gz}; best_pos[s & 1][wave] = gpos; }
    }
    __syncthreads();
    Best w = best[s & 1][lane & (W - 1)];   // repeated through the wave: the first row holds every wave's
    const int wp = best_pos[s & 1][lane & (W - 1)];
    const unsigned m = wave_max<1>(w.d);
    const unsigned long long cand = __ballot(w.d == m) & ((1ull << W) - 1);
    int l = __builtin_ctzll(cand);
    if (m && (cand & (cand - 1))) l = lane_of_least(cand, (int)order[wp]);
    if (m) {
      ox = lane_f(w.x, l); oy = lane_f(w.y, l); oz = lane_f(w.z, l);
      if (tid == l) out[s] = wp;   // a place in `order` for now: its translation would be waited for here
    } else {  // nothing but padding points: index 0, as the reference
      ox = p[0]; oy = p[1]; oz = p[2];
      if (tid == 0) out[s] = -1;
    }
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
__global__ __launch_bounds__(NTHREADS) void k_ball_query(int n, int m, float radius2, int nsample,
                                                         const float* __restrict__ new_xyz, const float* __restrict__ xyz,
                                                         int* __restrict__ idx) {
  const int b = blockIdx.y, lane = threadIdx.x & 63;
  const int j = blockIdx.x * (NTHREADS / 64) + (threadIdx.x >> 6);
  if (j >= m) return;  // whole wave
  const float* q = new_xyz + ((long)b * m + j) * 3;
  const float qx = q[0], qy = q[1], qz = q[2];
  const float* p = xyz + (long)b * n * 3;
  int* out = idx + ((long)b * m + j) * nsample;
  int cnt = 0, first = 0;
  for (int k0 = 0; k0 < n && cnt < nsample; k0 += 64) {
    const int k = k0 + lane;
    bool hit = false;
    if (k < n) {
      hit = sqdist(qx, qy, qz, p[k * 3], p[k * 3 + 1], p[k * 3 + 2]) < radius2;
    }
    const unsigned long long mask = __ballot(hit);
    if (mask == 0) continue;
    if (cnt == 0) first = k0 + __builtin_ctzll(mask);
    const int slot = cnt + __popcll(mask & ((1ull << lane) - 1ull));
    if (hit && slot < nsample) out[slot] = k;
    cnt += __popcll(mask);
  }
  if (cnt > nsample) cnt = nsample;
  for (int s = cnt + lane; s < nsample; s += 64) out[s] = first;  // first == 0 when nothing was found
}

// out[b][c][j][s] = points[b][c][idx[b][j][s]]   (one thread per output element)
__global__ __launch_bounds__(NTHREADS) void k_group_points(long total, int c, int n, int ms, const float* __restrict__ points,
                                                           const int* __restrict__ idx, float* __restrict__ out) {
  const long e = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= total) return;
  const int r = (int)(e % ms);
  const long bc = e / ms;
  const int b = (int)(bc / c);
  const int k = min(max(idx[(long)b * ms + r], 0), n - 1);  // a stray index must not leave the tensor
  out[e] = points[bc * n + k];
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

// 3 nearest known points of every unknown point: squared distances ascending, ties to the smaller index
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

int launch_fps(int b, int n, int npoint, const float* xyz, float* temp, int* idxs, hipStream_t st) {
#define FPS_GROUPS(W, S) hipLaunchKernelGGL((k_fps_groups<W, S>), dim3(b), dim3(64 * W), 0, st, n, npoint, xyz, idxs)
  // Eight waves up to 2048 points (fewer meet at the barrier: 0.73 against 0.78 us a draw at 2048), sixteen above (0.82
  // against 0.83 at 4096, 0.86 against 0.92 at 8192); slots just enough for n, every empty one costs 5 ns a draw.
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
  hipLaunchKernelGGL(k_ball_query, dim3((m + 3) / 4, b), dim3(NTHREADS), 0, st, n, m, radius * radius, nsample, new_xyz, xyz,
                     idx);
  return (int)hipGetLastError();
}
int launch_group_points(int b, int c, int n, int ms, const float* points, const int* idx, float* out, hipStream_t st) {
  const long total = (long)b * c * ms;
  hipLaunchKernelGGL(k_group_points, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, n, ms, points, idx, out);
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
  hipLaunchKernelGGL(k_three_nn, dim3((n + NTHREADS - 1) / NTHREADS, b), dim3(NTHREADS), 0, st, n, m, unknown, known, dist2,
                     idx);
  return (int)hipGetLastError();
}
int launch_three_interpolate(int b, int c, int m, int n, const float* points, const int* idx, const float* weight, float* out,
                             hipStream_t st) {
  const long total = (long)b * c * n;
  hipLaunchKernelGGL(k_three_interpolate, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, m, n, points, idx, weight,
                     out);
  return (int)hipGetLastError();
}
int launch_three_interpolate_grad(int b, int c, int n, int m, const float* grad_out, const int* idx, const float* weight,
                                  float* grad_points, hipStream_t st) {
  const long total = (long)b * c * n;
  hipLaunchKernelGGL(k_three_interpolate_grad, dim3(blocks_for(total)), dim3(NTHREADS), 0, st, total, c, n, m, grad_out, idx,
                     weight, grad_points);
  return (int)hipGetLastError();
}

}  // namespace issm
