// Box-to-point distance encoding and locality weight: the two (B, L, K) fields DEST computes right before the scan
// (gfx950).
//
// BoxDistFun.forward (models/dest_module.py:174-195): for every (key point l, query box k) and each of the box's 8
// corners, delta = corner - key, rotated in the x-y plane by the query angle, compressed by a signed log
// (sign(v) log2(|v| s + 1) / log2 8 / max_value), and used as the sampling position of a trilinear grid_sample
// (padding zeros, align_corners False) into a small learned table (C = 16 channels over D x H x W = 10^3 nodes); the
// 8 samples are summed into dist[b][l][k][0..15].  local_weight (dest_module.py:240-249):
// w[b][l][k] = exp(weight_dist * min(radius_k - |key_l - centre_k|, 0)).
// As tensor ops this materialises (B, 8K, L, 3) deltas several times and gathers 8 * 8 * 16 table entries per (l, k)
// from global memory.  Here the table (node-major: 16 channels of a node contiguous) lives in LDS, a wave owns one
// box (corners in scalar registers) and walks the key points with one (l, k) pair per lane, and the output row (16
// values) leaves as one contiguous store; no intermediate exists.  The backward is the table gradient only (corners are detached in the
// reference, key positions and angles are inputs): the same walk, scattering weight * ddist into an LDS copy of the
// table, then a sum of the per-workgroup copies.  The LDS copy is 64-bit fixed point (terms scaled by
// 2^34 / max|ddist|, found by a first pass): LDS integer atomics run about twice as fast as ds_add_f32 here, and
// integer sums do not depend on the order of the adds, so the gradient is reproducible bit for bit.
#include "box_dist_dev.h"

namespace issm {

// Locality weights: thread = (l, k) pair, k along the lanes (coalesced stores).
__global__ __launch_bounds__(NTHREADS) void k_box_dist_weights(BoxDistP p) {
  const Items it = my_items(p);
  float qx = 0.0f, qy = 0.0f, qz = 0.0f, radius = 0.0f;
  long cur = -1;
  for (long item = it.i0; item < it.i1; ++item) {
    const int l = (int)(item % p.L);
    const long bk = item / p.L;
    const int b = (int)(bk / it.kchunks), k = (int)(bk % it.kchunks) * NTHREADS + threadIdx.x;
    if (k >= p.K) continue;
    if (bk != cur) {
      if (p.qcenter) {
        const float* q = p.qcenter + ((long)b * p.K + k) * 3;
        qx = q[0]; qy = q[1]; qz = q[2];
        radius = p.radius[(long)b * p.K + k];
      } else {  // from the box: centre, radius = max(|size|, min_radius)
        const float* q = p.boxes + ((long)b * p.K + k) * 7;
        qx = q[0]; qy = q[1]; qz = q[2];
        radius = fmaxf(sqrtf(q[3] * q[3] + q[4] * q[4] + q[5] * q[5]), p.min_radius);
      }
      cur = bk;
    }
    const float* key = p.key + ((long)b * p.L + l) * 3;  // uniform
    const float ex = key[0] - qx, ey = key[1] - qy, ez = key[2] - qz;
    const float d = sqrtf(ex * ex + ey * ey + ez * ez);
    p.weights[((long)b * p.L + l) * p.K + k] = __expf(p.weight_dist * fminf(radius - d, 0.0f));
  }
}

template <bool BF>
__device__ __forceinline__ void store_dist(const BoxDistP& p, long o, const f4 (&acc)[4]) {
  if (BF) {
    uint4* dst = (uint4*)((uint16_t*)p.dist + o * BD_C);
    dst[0] = make_uint4(pack_bf16(acc[0].x, acc[0].y), pack_bf16(acc[0].z, acc[0].w), pack_bf16(acc[1].x, acc[1].y),
                        pack_bf16(acc[1].z, acc[1].w));
    dst[1] = make_uint4(pack_bf16(acc[2].x, acc[2].y), pack_bf16(acc[2].z, acc[2].w), pack_bf16(acc[3].x, acc[3].y),
                        pack_bf16(acc[3].z, acc[3].w));
  } else {
    f4* dst = (f4*)((float*)p.dist + o * BD_C);
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[j] = acc[j];
  }
}

__device__ __forceinline__ float wave_uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// dist: a wave owns one box (its corners and rotations in scalar registers) and up to BD_SEG key points, a lane one point
// at a time.  Pairs whose corners share a 3 x 3 x 3 window take the short path at once; the others (a box next to
// or around the point: about four in ten at detector scales) are queued in LDS and then walked corner by corner in
// full waves -- done in place, the long path would run for every wave with most lanes idle, and cost more than the
// rest together.  The sixteen waves of a workgroup own eight adjacent boxes, so a point's eight rows are neighbours in memory,
// and two segments of points each: four waves per SIMD on one table (vector issue bounds it, 83 M instructions; with two
// waves per SIMD their LDS reads were not hidden).  8 x 1024 points, 256 boxes: 219 -> 176 us; one scene, whose segments are
// shortened to 64 points so that all CUs have one (32 workgroups before): 209 -> 40 us.
// The table lies node-major in LDS with 20 floats from node to node: a lane reads its node's 16 channels as four
// 16-byte pieces, and with 16 floats per node the lanes of one read would meet in the 16 banks that (node mod 4)
// selects; 20 n mod 64 runs through all sixteen 4-bank groups as n does.
//
// AXES, calls that nothing is differentiated through: boxes that stand along the axes, under no rotation.  The eight corners are
// two positions per axis, so the sum of their trilinear weights is a product of three sums over an axis' positions: at most four nodes
// an axis, 6 logarithms a pair instead of 24, no queue (all pairs, whether the box is next to the point or around it).  Taken by a
// wave whose box is such a one, for finite points and a finite table.  Bound by the LDS reads, 64 bytes a node and lane; a lane
// leaves out the nodes of weight zero (outside the table, or the other position's): with all of them read, points in random order lost
// to the form by corners.  A call of the encoding, 256 boxes, 1024 points a scene, bf16, by corners, with every node read and like this: one scene, in the
// order of a Hilbert curve 49.7, 37.2 and 34.9 us, in random order 50.5, 44.4 and 36.1; eight 171, 103 and 90, 184, 190 and 113.  Boxes that are
// turned pay 0.6 us a launch for the look at them (47 and 201 us).
// As accurate, but rounded elsewhere, and an encoding that differs in the last bit of one value in ten thousand moves entries of a
// gradient behind six bf16 layers by up to 0.48 of their mean square: training keeps the sums it had.
// In training such a box's corners still enter one by one, the same operations in the same order, but from the two positions an axis has
// (corner_window_axes; in the queue too): 6 logarithms and 36 products of two axes a pair instead of 24 and 72.  8 x 1024 points, 256 boxes, bf16 162
// -> 139 us, the same values.  (Loops of their own: with both forms in one step the kernel spilled 92 bytes a lane.)
constexpr int BD_SEG = 512;     // points per wave at most
constexpr int BD_FWD_T = 1024;  // 16 waves = 8 adjacent boxes x 2 segments per workgroup, one workgroup (96 KB of LDS) per CU
constexpr int BD_NS = 20;      // floats from node to node

// An axis of a box along the axes: the nodes its two positions lie between and their summed weights; nodes outside the table
// and those the other position has already have weight zero.
struct AxisNodes {
  int node[4];
  float w[4];
};
__device__ __forceinline__ AxisNodes axis_nodes(float p0, float p1, int n, int stride) {
  const float g0 = floorf(p0), g1 = floorf(p1), a0 = p0 - g0, a1 = p1 - g1;
  const int i0 = (int)g0, i1 = (int)g1;
  const bool same = i1 == i0, up = i1 == i0 + 1, down = i1 + 1 == i0;
  AxisNodes a;
  a.node[0] = i0;
  a.w[0] = (1.0f - a0) + (same ? 1.0f - a1 : down ? a1 : 0.0f);
  a.node[1] = i0 + 1;
  a.w[1] = a0 + (same ? a1 : up ? 1.0f - a1 : 0.0f);
  a.node[2] = up ? i1 + 1 : i1;
  a.w[2] = same ? 0.0f : up ? a1 : 1.0f - a1;
  a.node[3] = i1 + 1;
  a.w[3] = same || up || down ? 0.0f : a1;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool in = a.node[e] >= 0 && a.node[e] < n;
    a.node[e] = in ? a.node[e] * stride : 0;
    a.w[e] = in ? a.w[e] : 0.0f;
  }
  return a;
}
template <bool BF, bool AXES>
__global__ __launch_bounds__(BD_FWD_T) void k_box_dist_fwd(BoxDistP p, int seg_points) {
  __shared__ __attribute__((aligned(16))) float tab[BD_MAXCELLS * BD_NS];
  __shared__ unsigned short queue[BD_FWD_T / 64][BD_SEG];
  __shared__ int queue_len[BD_FWD_T / 64], odd_of[BD_FWD_T / 64];
  const int cells = p.D * p.H * p.W;
  bool odd = false;   // AXES: some value of the table is not finite (odd_of: of a wave's share of it)
  for (int e = threadIdx.x; e < cells * BD_C; e += BD_FWD_T) {
    const int ch = e / cells, cell = e - ch * cells;
    const float v = p.table[e];
    tab[cell * BD_NS + ch] = v;
    if constexpr (AXES) odd |= !finite_(v);
  }
  if constexpr (AXES) odd_of[threadIdx.x >> 6] = __ballot(odd) != 0ull;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kgroups = (p.K + 7) / 8, npair = (p.L + 2 * seg_points - 1) / (2 * seg_points);
  const int kgroup = blockIdx.x % kgroups, bs = blockIdx.x / kgroups;
  const int b = bs / npair, k = kgroup * 8 + (wave & 7);
  const int l0 = (2 * (bs % npair) + (wave >> 3)) * seg_points, n = min(seg_points, p.L - l0);
  const bool live = k < p.K;  // uniform per wave (n may be 0 or less)
  const float scale = 1.0f / (3.0f * p.max_value);
  BoxLane bx;
  int queued = 0;
  if (live) {
    load_box(p, b, k, bx);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      bx.cx[c] = wave_uniform(bx.cx[c]); bx.cy[c] = wave_uniform(bx.cy[c]); bx.cz[c] = wave_uniform(bx.cz[c]);
      bx.cs[c] = wave_uniform(bx.cs[c]); bx.sn[c] = wave_uniform(bx.sn[c]);
    }
    int base = 0;
    const bool aligned = along_axes(bx);   // uniform
    bool axes = AXES && aligned;
    if (axes) {
#pragma unroll
      for (int w = 0; w < BD_FWD_T / 64; ++w) axes = axes && __builtin_amdgcn_readfirstlane(odd_of[w]) == 0;
    }
    if (axes) {   // uniform
      const float x0 = bx.cx[0], x1 = bx.cx[2], y0 = bx.cy[0], y1 = bx.cy[1], z0 = bx.cz[0], z1 = bx.cz[4];
#pragma unroll 1
      for (; base < n; base += 64) {
        const int li = base + lane;
        const float* key = p.key + ((long)b * p.L + l0 + min(li, n - 1)) * 3;
        const float kx = key[0], ky = key[1], kz = key[2];
        if (__ballot(!(finite_(kx) && finite_(ky) && finite_(kz))) != 0ull) break;   // (this and what follows: below)
        const AxisNodes ax = axis_nodes(node_pos(x0 - kx, p.log_scale, scale, p.W), node_pos(x1 - kx, p.log_scale, scale, p.W), p.W, BD_NS),
                        ay = axis_nodes(node_pos(y0 - ky, p.log_scale, scale, p.H), node_pos(y1 - ky, p.log_scale, scale, p.H), p.H, p.W * BD_NS);
        AxisNodes az = axis_nodes(node_pos(z0 - kz, p.log_scale, scale, p.D), node_pos(z1 - kz, p.log_scale, scale, p.D), p.D, p.H * p.W * BD_NS);
        f4 acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
        const bool x2 = __ballot(ax.w[2] != 0.0f) != 0ull, x3 = __ballot(ax.w[3] != 0.0f) != 0ull;
#pragma unroll 1
        for (int k3 = 0; k3 < 4; ++k3) {   // (always entry 0 of az, whose entries move up: registers are not indexed)
#pragma unroll
          for (int i3 = 0; i3 < 4; ++i3) {
            const float zy = az.w[0] * ay.w[i3];
            if (__ballot(zy != 0.0f) == 0ull) continue;
            const float* row = tab + az.node[0] + ay.node[i3];
            auto node = [&](int j3) {
              const f4* src = (const f4*)(row + ax.node[j3]);
              const float w = zy * ax.w[j3];
              if (w != 0.0f) {
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] += w * src[j];
              }
            };
            node(0);
            node(1);
            if (x2) node(2);
            if (x3) node(3);
          }
#pragma unroll
          for (int e = 0; e < 3; ++e) az.node[e] = az.node[e + 1], az.w[e] = az.w[e + 1];
        }
        if (li < n) store_dist<BF>(p, ((long)b * p.L + l0 + li) * p.K + k, acc);
      }
    }
    // a step's points: those with a window at once, the others into the queue
    auto step = [&](auto window) __attribute__((always_inline)) {
      const int li = base + lane;
      const bool valid = li < n;
      const float* key = p.key + ((long)b * p.L + l0 + (valid ? li : n - 1)) * 3;
      const float kx = key[0], ky = key[1], kz = key[2];
      Window win;
      const int one_window = window(kx, ky, kz, win);
      if (one_window < 0) return false;   // uniform
      if (valid && one_window) {
        f4 acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
        for_window(p, win, [&](int off, float w) {
          const f4* src = (const f4*)(tab + off);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] += w * src[j];
        }, BD_NS);
        store_dist<BF>(p, ((long)b * p.L + l0 + li) * p.K + k, acc);
      }
      const unsigned long long rest = __ballot(valid && !one_window);
      if (valid && !one_window) queue[wave][queued + __popcll(rest & ((1ull << lane) - 1ull))] = (unsigned short)li;
      queued += __popcll(rest);
      return true;
    };
    if (aligned) {
#pragma unroll 1
      for (; base < n; base += 64)
        if (!step([&](float kx, float ky, float kz, Window& win) -> int {
              if (__ballot(!(finite_(kx) && finite_(ky) && finite_(kz))) != 0ull) return -1;   // (this and what follows: below)
              return corner_window_axes(p, bx, kx, ky, kz, scale, win);
            })) break;
    }
#pragma unroll 1
    for (; base < n; base += 64) step([&](float kx, float ky, float kz, Window& win) -> int { return corner_window(p, bx, kx, ky, kz, scale, win); });
  }
  if (lane == 0) queue_len[wave] = queued;
  __syncthreads();
  if (!live) return;
  // the box's two waves take the points both have queued in turn, 64 at a time: one wave that is not full instead of two, and both
  // end together (eight scenes, points in the order of a Hilbert curve, bf16: 176 -> 163 us; in random order 178 either way, fp32
  // 193 -> 186; one scene, 26 points a queue, 39.5 either way)
  const int qa = queue_len[wave & 7], all = qa + queue_len[(wave & 7) + 8], la = 2 * (bs % npair) * seg_points;
  for (int i = (wave >> 3) * 64 + lane; i < all; i += 128) {
    const int l = i < qa ? la + queue[wave & 7][i] : la + seg_points + queue[(wave & 7) + 8][i - qa];
    const float* key = p.key + ((long)b * p.L + l) * 3;
    const float kx = key[0], ky = key[1], kz = key[2];
    f4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto corner = [&](float x, float y, float z) __attribute__((always_inline)) {
      Tri t;
      trilinear(p, x, y, z, t, BD_NS);
#pragma unroll
      for (int n8 = 0; n8 < 8; ++n8) {
        const f4* src = (const f4*)(tab + t.off[n8]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] += t.w[n8] * src[j];
      }
    };
    if (along_axes(bx) && __ballot(!(finite_(kx) && finite_(ky) && finite_(kz))) == 0ull) {   // uniform; the same sums from two positions an axis
      const float x0 = node_pos(bx.cx[0] - kx, p.log_scale, scale, p.W), x1 = node_pos(bx.cx[2] - kx, p.log_scale, scale, p.W),
                  y0 = node_pos(bx.cy[0] - ky, p.log_scale, scale, p.H), y1 = node_pos(bx.cy[1] - ky, p.log_scale, scale, p.H),
                  z0 = node_pos(bx.cz[0] - kz, p.log_scale, scale, p.D), z1 = node_pos(bx.cz[4] - kz, p.log_scale, scale, p.D);
#pragma unroll 1
      for (int c = 0; c < 8; ++c) corner(c & 2 ? x1 : x0, (c ^ (c >> 1)) & 1 ? y1 : y0, c & 4 ? z1 : z0);
    } else {
      // A rolled loop that always works on slot 0 and then rotates the box's registers by one corner: fully unrolled,
      // the compiler issues the LDS reads of all 8 corners first and spills them.
#pragma unroll 1
      for (int c = 0; c < 8; ++c) {
        const float dx = bx.cx[0] - kx, dy = bx.cy[0] - ky, dz = bx.cz[0] - kz;
        const float rx = dx * bx.cs[0] - dy * bx.sn[0], ry = dx * bx.sn[0] + dy * bx.cs[0];
        corner(node_pos(rx, p.log_scale, scale, p.W), node_pos(ry, p.log_scale, scale, p.H), node_pos(dz, p.log_scale, scale, p.D));
        rotate_box(bx);
      }
    }
    store_dist<BF>(p, ((long)b * p.L + l) * p.K + k, acc);
  }
}

// The learned table without a gradient: Linear(3, hidden), ReLU, Linear(hidden, 16) at the nodes of the lattice (dest_module.py:191),
// rounded where the modules round (bf16: the hidden values and the results; fp32 sums).  16 nodes a workgroup, a (node, channel)
// pair a thread; the hidden values and the second weights lie in LDS.  2.4 M products at 1000 nodes and 128 hidden: bound by the
// launch and one trip to memory.  As modules it is seven launches, 28 us and 70 us of host time; this takes 5 us.
template <bool BF>
__global__ __launch_bounds__(NTHREADS) void k_box_table(BoxTableP p) {
  extern __shared__ float box_table_lds[];
  const int R = p.hidden, ld = R + 1, node0 = blockIdx.x * 16;
  float *h = box_table_lds, *w2 = box_table_lds + 16 * ld;
  constexpr int io = BF ? 1 : 0;
  __shared__ float xyz[16][3];
  if (threadIdx.x < 48) {
    const int i = threadIdx.x / 3, c = threadIdx.x - 3 * i;
    const float x = ldv(p.coords, 3L * min(node0 + i, p.nodes - 1) + c, p.coords_dtype);
    xyz[i][c] = BF ? bf16_to_f(f_to_bf16(x)) : x;
  }
  // a thread takes every 16th hidden value of its row: of W2 (channels), then of the hidden values (nodes)
  const int row = threadIdx.x >> 4;
#pragma unroll 8
  for (int r = threadIdx.x & 15; r < R; r += 16) w2[row * ld + r] = ldv(p.w2, (long)row * R + r, io);
  __syncthreads();
#pragma unroll 8
  for (int r = threadIdx.x & 15; r < R; r += 16) {
    float v = xyz[row][0] * ldv(p.w1, 3L * r, io);
    v = fmaf(xyz[row][1], ldv(p.w1, 3L * r + 1, io), v);
    v = fmaf(xyz[row][2], ldv(p.w1, 3L * r + 2, io), v) + ldv(p.b1, r, io);
    if (BF) v = bf16_to_f(f_to_bf16(v));
    h[row * ld + r] = v < 0.0f ? 0.0f : v;   // (NaN stays)
  }
  __syncthreads();
  const int i = threadIdx.x & 15, ch = threadIdx.x >> 4;
  float v = 0.0f;
#pragma unroll 8
  for (int r = 0; r < R; ++r) v = fmaf(h[i * ld + r], w2[ch * ld + r], v);
  if (BF) v = bf16_to_f(f_to_bf16(v));
  if (node0 + i < p.nodes) p.table[(long)ch * p.nodes + node0 + i] = v;
}

int launch_box_table(const BoxTableP& p, hipStream_t st) {
  const dim3 g((unsigned)((p.nodes + 15) / 16)), b(NTHREADS);
  const size_t lds = (size_t)2 * 16 * (p.hidden + 1) * sizeof(float);
  if (p.dtype) hipLaunchKernelGGL(k_box_table<true>, g, b, lds, st, p);
  else hipLaunchKernelGGL(k_box_table<false>, g, b, lds, st, p);
  return (int)hipGetLastError();
}

// The table's backward: a workgroup has a hidden value, its threads take every NTHREADS-th node, whose hidden value is computed again.  Few MB and
// products: bound by the launch, a trip to memory and the 20 sums.  As modules it was nine launches and 90 us at 1000 nodes and 128
// hidden values; this takes 10.7.
template <bool BF>
__global__ __launch_bounds__(NTHREADS) void k_box_table_bwd(BoxTableP p, const float* __restrict__ dtable, void* dw1, void* db1, void* dw2) {
  constexpr int io = BF ? 1 : 0, NS_ = BD_C + 4;   // sums: of W2's channels, b1, W1's three
  __shared__ float red[NTHREADS / 64][NS_];
  const int r = blockIdx.x, lane = threadIdx.x & 63;
  const float wx = ldv(p.w1, 3L * r, io), wy = ldv(p.w1, 3L * r + 1, io), wz = ldv(p.w1, 3L * r + 2, io), b1 = ldv(p.b1, r, io);
  float w2[BD_C], sum[NS_];
#pragma unroll
  for (int c = 0; c < BD_C; ++c) w2[c] = ldv(p.w2, (long)c * p.hidden + r, io);
#pragma unroll
  for (int c = 0; c < NS_; ++c) sum[c] = 0.0f;
#pragma unroll 2
  for (int n = threadIdx.x; n < p.nodes; n += NTHREADS) {
    float x[3], g[BD_C];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = ldv(p.coords, 3L * n + c, p.coords_dtype);
#pragma unroll
    for (int c = 0; c < BD_C; ++c) g[c] = dtable[(long)c * p.nodes + n];
    if (BF)
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] = bf16_round(x[c]);
    float h = fmaf(wz, x[2], fmaf(wy, x[1], wx * x[0])) + b1;   // (as k_box_table)
    if (BF) h = bf16_round(h);
    h = h < 0.0f ? 0.0f : h;
    float dh = 0.0f;
#pragma unroll
    for (int c = 0; c < BD_C; ++c) {
      dh = fmaf(g[c], w2[c], dh);
      sum[c] = fmaf(g[c], h, sum[c]);
    }
    dh = h <= 0.0f ? 0.0f : dh;   // (of NaN the gradient passes, as the module's does)
    sum[BD_C] += dh;
#pragma unroll
    for (int c = 0; c < 3; ++c) sum[BD_C + 1 + c] = fmaf(dh, x[c], sum[BD_C + 1 + c]);
  }
#pragma unroll
  for (int c = 0; c < NS_; ++c) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum[c] += __shfl_xor(sum[c], o, 64);
    if (lane == 0) red[threadIdx.x >> 6][c] = sum[c];
  }
  __syncthreads();
  const int c = threadIdx.x;
  if (c >= NS_) return;
  const float v = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  if (c < BD_C) stv(dw2, (long)c * p.hidden + r, io, v);
  else if (c == BD_C) stv(db1, r, io, v);
  else stv(dw1, 3L * r + c - BD_C - 1, io, v);
}

int launch_box_table_bwd(const BoxTableP& p, const float* dtable, void* dw1, void* db1, void* dw2, hipStream_t st) {
  const dim3 g((unsigned)p.hidden), b(NTHREADS);
  if (p.dtype) hipLaunchKernelGGL(k_box_table_bwd<true>, g, b, 0, st, p, dtable, dw1, db1, dw2);
  else hipLaunchKernelGGL(k_box_table_bwd<false>, g, b, 0, st, p, dtable, dw1, db1, dw2);
  return (int)hipGetLastError();
}

__global__ void k_box_dist_clear(unsigned* scal) { scal[0] = 0u; }

// max |ddist| (bit pattern of a non-negative float orders like the unsigned integer)
template <bool BF>
__global__ __launch_bounds__(NTHREADS) void k_box_dist_gmax(BoxDistP p, unsigned* scal) {
  const long n = (long)p.B * p.L * p.K * BD_C;
  float m = 0.0f;
  for (long e = ((long)blockIdx.x * NTHREADS + threadIdx.x) * 8; e < n; e += (long)gridDim.x * NTHREADS * 8) {
    if (BF) {
      const uint4 v = *(const uint4*)((const uint16_t*)p.ddist + e);
      const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        m = fmaxf(m, fmaxf(fabsf(__uint_as_float(w[j] << 16)), fabsf(__uint_as_float(w[j] & 0xffff0000u))));
    } else {
      const f4 a = *(const f4*)((const float*)p.ddist + e), c = *(const f4*)((const float*)p.ddist + e + 4);
      m = fmaxf(m, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
      m = fmaxf(m, fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w))));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0 && m > 0.0f && m == m) atomicMax(scal, __float_as_uint(m));
}

// Table gradient: partial[wg][cell][ch] = sum over the workgroup's (l, k) pairs and corners of weight * ddist.
template <bool BF>
__global__ __launch_bounds__(NTHREADS) void k_box_dist_bwd(BoxDistP p) {
  __shared__ __attribute__((aligned(16))) unsigned long long tab[BD_MAXCELLS * BD_C];  // 128 KB: one workgroup per CU
  const int cells = p.D * p.H * p.W;
  for (int e = threadIdx.x; e < cells * BD_C; e += NTHREADS) tab[e] = 0ull;
  __syncthreads();
  const float fx_scale = bd_scale((const unsigned*)p.partial);
  const Items it = my_items(p);
  const float scale = 1.0f / (3.0f * p.max_value);
  int rot[BD_C];
#pragma unroll
  for (int j = 0; j < BD_C; ++j) rot[j] = (j + threadIdx.x) & 15;
  BoxLane bx;
  long cur = -1;
  for (long item = it.i0; item < it.i1; ++item) {
    const int l = (int)(item % p.L);
    const long bk = item / p.L;
    const int b = (int)(bk / it.kchunks), k = (int)(bk % it.kchunks) * NTHREADS + threadIdx.x;
    if (k >= p.K) continue;
    if (bk != cur) {
      load_box(p, b, k, bx);
      cur = bk;
    }
    const float* key = p.key + ((long)b * p.L + l) * 3;
    const float kx = key[0], ky = key[1], kz = key[2];
    const long o = ((long)b * p.L + l) * p.K + k;
    float g[BD_C];
    if (BF) {
      const uint4* src = (const uint4*)((const uint16_t*)p.ddist + o * BD_C);
      const uint4 a = src[0], c = src[1];
      const unsigned w[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        g[2 * j] = __uint_as_float(w[j] << 16);
        g[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
      }
    } else {
      const f4* src = (const f4*)((const float*)p.ddist + o * BD_C);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f4 v = src[j];
        g[4 * j] = v.x; g[4 * j + 1] = v.y; g[4 * j + 2] = v.z; g[4 * j + 3] = v.w;
      }
    }
#pragma unroll
    for (int j = 0; j < BD_C; ++j) g[j] *= fx_scale;
    // Lane r adds channel (j + r) mod 16 at step j.  Samples crowd into few nodes (the signed log maps most
    // distances near +-1), so many lanes of a wave hit the same node at once: with every lane on channel j that is
    // one LDS address and the adds serialise; rotated, the lanes of a node spread over its 16 channels.
#pragma unroll
    for (int bit = 8; bit >= 1; bit >>= 1) {
      const bool on = (threadIdx.x & bit) != 0;
      float t[BD_C];
#pragma unroll
      for (int j = 0; j < BD_C; ++j) t[j] = on ? g[(j + bit) & 15] : g[j];
#pragma unroll
      for (int j = 0; j < BD_C; ++j) g[j] = t[j];
    }
    Window win;
    if (corner_window(p, bx, kx, ky, kz, scale, win)) {
      for_window(p, win, [&](int off, float w) {
        unsigned long long* dst = tab + off;
#pragma unroll
        for (int j = 0; j < BD_C; ++j) atomicAdd(dst + rot[j], (unsigned long long)__float2ll_rn(w * g[j]));
      });
    } else {
#pragma unroll 1
      for (int c = 0; c < 8; ++c) {
        const float dx = bx.cx[0] - kx, dy = bx.cy[0] - ky, dz = bx.cz[0] - kz;
        const float rx = dx * bx.cs[0] - dy * bx.sn[0], ry = dx * bx.sn[0] + dy * bx.cs[0];
        Tri t;
        trilinear(p, node_pos(rx, p.log_scale, scale, p.W), node_pos(ry, p.log_scale, scale, p.H),
                  node_pos(dz, p.log_scale, scale, p.D), t);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          if (t.w[n] != 0.0f) {
            unsigned long long* dst = tab + t.off[n];
#pragma unroll
            for (int j = 0; j < BD_C; ++j) atomicAdd(dst + rot[j], (unsigned long long)__float2ll_rn(t.w[n] * g[j]));
          }
        }
        rotate_box(bx);
      }
    }
  }
  __syncthreads();
  unsigned long long* out = (unsigned long long*)p.partial + 2 + (long)blockIdx.x * cells * BD_C;
  for (int e = threadIdx.x; e < cells * BD_C; e += NTHREADS) out[e] = tab[e];
}

// dtable[ch][cell] = (sum over workgroups of partial[wg][cell][ch], exact in 64 bits) / scale
__global__ __launch_bounds__(NTHREADS) void k_box_dist_dtable(BoxDistP p) {
  const int cells = p.D * p.H * p.W;
  const int e = blockIdx.x * NTHREADS + threadIdx.x;  // e = cell * 16 + ch
  if (e >= cells * BD_C) return;
  const long long* part = (const long long*)p.partial + 2;
  long long a = 0;
  for (int w = 0; w < p.nwg_bwd; ++w) a += part[(long)w * cells * BD_C + e];
  const int cell = e / BD_C, ch = e % BD_C;
  p.dtable[(long)ch * cells + cell] = (float)((double)a / (double)bd_scale((const unsigned*)p.partial));
}

int box_dist_workgroups(int B, int L, int K) {
  const long items = (long)B * ((K + NTHREADS - 1) / NTHREADS) * L;
  return (int)(items < 512 ? items : 512);  // forward: two 64 KB workgroups per CU
}
int box_dist_bwd_workgroups(int B, int L, int K) {
  const long items = (long)B * ((K + NTHREADS - 1) / NTHREADS) * L;
  return (int)(items < 256 ? items : 256);  // backward: one 128 KB workgroup per CU
}

int launch_box_dist_fwd(const BoxDistP& p, bool only, hipStream_t st) {
  const dim3 b(NTHREADS);
  if (p.dist) {
    // segments of whole waves, as long as the queue allows but no longer than leaves every CU (256) a workgroup
    const long rows = (long)p.B * ((p.K + 7) / 8), want = (256 + rows - 1) / rows;
    const int half = (int)((p.L + 2 * want - 1) / (2 * want)), seg = half >= BD_SEG ? BD_SEG : (half + 63) / 64 * 64;
    const dim3 g((unsigned)(rows * ((p.L + 2 * seg - 1) / (2 * seg))));
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, dim3(BD_FWD_T), 0, st, p, seg); };
    if (p.dtype) only ? go(&k_box_dist_fwd<true, true>) : go(&k_box_dist_fwd<true, false>);
    else only ? go(&k_box_dist_fwd<false, true>) : go(&k_box_dist_fwd<false, false>);
  }
  if (p.weights) hipLaunchKernelGGL(k_box_dist_weights, dim3(p.nwg), b, 0, st, p);
  return (int)hipGetLastError();
}

int launch_box_dist_bwd_sorted(const BoxDistP& p, hipStream_t st);
long box_dist_sorted_scratch_bytes(int B, int L, int K, int D, int H, int W);

// few pairs: scatter with LDS atomics (one launch of work); many pairs: sort by window, then dense sums
constexpr long BD_SORT_MIN_PAIRS = 1 << 16;

long box_dist_bwd_scratch_bytes(int B, int L, int K, int D, int H, int W) {
  const long atomic_path = 16 + (long)box_dist_bwd_workgroups(B, L, K) * D * H * W * BD_C * 8;
  if ((long)B * L * K < BD_SORT_MIN_PAIRS) return atomic_path;
  const long sorted_path = box_dist_sorted_scratch_bytes(B, L, K, D, H, W);
  return sorted_path > atomic_path ? sorted_path : atomic_path;
}

int launch_box_dist_bwd(const BoxDistP& p, hipStream_t st) {
  if ((long)p.B * p.L * p.K >= BD_SORT_MIN_PAIRS) return launch_box_dist_bwd_sorted(p, st);
  const dim3 g(p.nwg_bwd), b(NTHREADS);
  unsigned* scal = (unsigned*)p.partial;
  hipLaunchKernelGGL(k_box_dist_clear, dim3(1), dim3(1), 0, st, scal);
  if (p.dtype) hipLaunchKernelGGL(k_box_dist_gmax<true>, dim3(512), b, 0, st, p, scal);
  else hipLaunchKernelGGL(k_box_dist_gmax<false>, dim3(512), b, 0, st, p, scal);
  if (p.dtype) hipLaunchKernelGGL(k_box_dist_bwd<true>, g, b, 0, st, p);
  else hipLaunchKernelGGL(k_box_dist_bwd<false>, g, b, 0, st, p);
  int e = (int)hipGetLastError();
  if (e) return e;
  const int n = p.D * p.H * p.W * BD_C;
  hipLaunchKernelGGL(k_box_dist_dtable, dim3((n + NTHREADS - 1) / NTHREADS), b, 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace issm
