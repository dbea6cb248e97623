// Inter-chunk recurrences of the ISSM scan (gfx950), bound by HBM: every chunk's state is read once and written once.
//
//   forward:   H_0 = h0,          H_(c+1)  = exp(cs_last_c) H_c  + S_c    slot c of `states`:  S_c in, H_c out; slot nc: H_nc
//   backward:  dS_(nc-1) = dfinal, dS_(c-1) = exp(cs_last_c) dS_c + dH_c   slot c of `dstates`: dH_c in, dS_c out
//
// The same recurrence, walked from the other end.  It is element-wise, so a thread carries 4 adjacent columns of one state row
// through all chunks, and a wave's accesses are whole rows (1 KB at 256 columns).  (The backward pass once also read the forward's
// states, half as much again, for the column sums g = sum_p dS_c H_(c+1) that d/d(cs) needs, in slices of 32 or 64 columns by all
// rows with the rows' sums through LDS.  The chunk backward now takes g from what it has in registers, see k_bwd_tile.
// Launched over and over on the same buffers, backward, 2 x 16384 tokens, 8 heads x 32, 256 states: 109 -> 47 us, 5.8 TB/s (inside a
// training step, where the buffers come from HBM, 62, 4.3 TB/s); 8 x 1024, both directions: 32 -> 26; forward, inside a step, 16 x 2048, 16 heads
// x 64, 512 states, both directions: 0.93 ms, 4.6 TB/s.)
#include "issm_dev.h"

namespace issm {

// Where a recurrence starts, ends and walks.  BACK: the backward one.
template <bool BACK>
struct Pass {
  const void* first;   // fp32 or bf16 (forward), row strides s0, s1, s2; may be NULL: zero
  long s0, s1, s2;
  int first_dt;
  float* slots;        // the first chunk's slot of (bt, h)
  const float* decay;
  float* last;         // what the recurrence ends in, (P, N); may be NULL
  __device__ __forceinline__ Pass(const KP& p, float* st, const float* cs_last, float* dh0_dir, int bt, int h) {
    const int b = bt / p.ndir, dir = bt % p.ndir;
    const long slab = (long)p.P * p.N, at = ((long)b * p.H + h) * slab;
    if constexpr (BACK) {
      first = p.dfinal[dir];
      s0 = p.H * slab, s1 = slab, s2 = p.N, first_dt = 0;
      slots = st + dst_off(p, bt, p.nc - 1, h);
      decay = cs_last + vec_off(p, bt, p.nc - 1, h);
      last = dh0_dir + (long)dir * p.B * p.H * slab + at;
    } else {
      first = p.h0.ptr;
      s0 = p.h0.s0, s1 = p.h0.s1, s2 = p.h0.s2, first_dt = p.h0_dt;
      slots = st + st_off(p, bt, 0, h);
      decay = cs_last + vec_off(p, bt, 0, h);
      last = p.final_states[dir] ? p.final_states[dir] + at : nullptr;
    }
    if (first) s0 = b * s0 + h * s1;
  }
  __device__ __forceinline__ float start(int pp, int n) const { return first ? ldv(first, s0 + pp * s2 + n, first_dt) : 0.0f; }
};

// The recurrence without any conditional access in its loop: the operands of the next D chunks are always requested (near the end
// the last chunk's again: in range, unused), so the compiler can count the loads in flight and never waits for all of them; with
// loads inside branches it did, once per chunk.  D = 8 when few threads walk many chunks (memory latency sets the pace there),
// otherwise 4.
// TAIL (N >= 4, not a multiple of 4; accesses at any float): the last thread of a row works on columns N - 4 .. N - 1 and
// stores only those its neighbour does not own (what it computes for the others may read the neighbour's results and is
// dropped).  8 x 1024 tokens, N = 250: 30.3 us with per-element guards, as fast as N = 256 without.
template <int D, bool TAIL, bool BACK>
__global__ __launch_bounds__(NTHREADS) void k_state_pass(KP p, float* __restrict__ states, const float* __restrict__ cs_last,
                                                         float* __restrict__ dh0_dir) {
  warm_args();
  const int nq = (p.N + 3) >> 2;
  const long total = (long)p.B * p.ndir * p.H * p.P * nq;
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= total) return;
  int q, pp, h, bt;
  if (total < (1L << 31)) {
    unsigned r = (unsigned)id;
    q = (int)p.by_quads(r);
    pp = (int)p.by_P(r);
    h = (int)p.by_H(r);
    bt = (int)r;
  } else {
    q = id % nq;
    const long r = id / nq;
    pp = r % p.P;
    h = r / p.P % p.H;
    bt = r / p.P / p.H;
  }
  const int n = TAIL ? min(q * 4, p.N - 4) : q * 4, skip = q * 4 - n;   // skip: columns of the thread that are its neighbour's
  auto ld = [](const float* a) -> f4 {
    if constexpr (TAIL) return ld_f4_any(a);
    else return *(const f4*)a;
  };
  auto put = [&](float* a, f4 v) {
    if constexpr (!TAIL) {
      *(f4*)a = v;
    } else if (skip == 0) {
      st_f4_any(a, v);
    } else {
#pragma unroll
      for (int j = 1; j < 4; ++j)
        if (j >= skip) a[j] = v[j];
    }
  };
  const Pass<BACK> w(p, states, cs_last, dh0_dir, bt, h);
  f4 st;
#pragma unroll
  for (int j = 0; j < 4; ++j) st[j] = w.start(pp, n + j);
  const long cstride = (BACK ? -1 : 1) * (long)p.H * p.P * p.N, dstride = (BACK ? -1 : 1) * (long)p.H * p.N;
  float* sp = w.slots + (long)pp * p.N + n;
  // step c lives in slot c % D; the loop is unrolled over the D slots so that none is ever moved (a register copy
  // would have to wait for the load that fills it)
  const float* sp0 = sp;
  const float* cl0 = w.decay + n;
  f4 t[D], d[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const int ci = min(i, p.nc - 1);
    t[i] = ld(sp0 + ci * cstride);
    d[i] = ld(cl0 + ci * dstride);
  }
  int c = 0;
  for (; c + D <= p.nc; c += D) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const f4 tt = t[i], dd = d[i];
      const int cn = min(c + i + D, p.nc - 1);
      t[i] = ld(sp0 + cn * cstride);
      d[i] = ld(cl0 + cn * dstride);
      put(sp, st);
#pragma unroll
      for (int j = 0; j < 4; ++j) st[j] = __expf(dd[j]) * st[j] + tt[j];
      sp += cstride;
    }
  }
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    if (c + i < p.nc) {  // uniform: the last nc % D chunks
      put(sp, st);
#pragma unroll
      for (int j = 0; j < 4; ++j) st[j] = __expf(d[i][j]) * st[j] + t[i][j];
      sp += cstride;
    }
  if constexpr (!BACK) put(sp, st);  // slot nc keeps the final state for the backward pass
  if (w.last) put(w.last + (long)pp * p.N + n, st);
}

// The recurrence for N < 4: thread = one element, scalar accesses.
template <bool BACK>
__global__ __launch_bounds__(NTHREADS) void k_state_pass_narrow(KP p, float* __restrict__ states,
                                                                const float* __restrict__ cs_last, float* __restrict__ dh0_dir) {
  const long total = (long)p.B * p.ndir * p.H * p.P * p.N;
  const long id = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (id >= total) return;
  const int n = id % p.N;
  long r = id / p.N;
  const int pp = r % p.P;
  r /= p.P;
  const int h = r % p.H;
  const Pass<BACK> w(p, states, cs_last, dh0_dir, r / p.H, h);
  const long cstride = (BACK ? -1 : 1) * (long)p.H * p.P * p.N, dstride = (BACK ? -1 : 1) * (long)p.H * p.N;
  float* sp = w.slots + (long)pp * p.N + n;
  const float* cl = w.decay + n;
  float st = w.start(pp, n);
  for (int c = 0; c < p.nc; ++c) {
    const float s = *sp, d = *cl;
    *sp = st;
    st = __expf(d) * st + s;
    sp += cstride;
    cl += dstride;
  }
  if constexpr (!BACK) *sp = st;
  if (w.last) w.last[(long)pp * p.N + n] = st;
}

// g_c[n] = sum_p dS_c[p,n] H_(c+1)[p,n], for callers of the stage entry points that ask for it: thread = column of a unit.
__global__ __launch_bounds__(NTHREADS) void k_state_sums(KP p, const float* __restrict__ states, const float* __restrict__ dstates,
                                                         float* __restrict__ g_last) {
  const long total = (long)p.B * p.ndir * p.nc * p.H * p.N;
  const long id = (long)blockIdx.x * NTHREADS + threadIdx.x;
  if (id >= total) return;
  const int n = id % p.N;
  long r = id / p.N;
  const int h = r % p.H;
  r /= p.H;
  const int c = r % p.nc, bt = r / p.nc;
  const float* hp = states + st_off(p, bt, c + 1, h) + n;
  const float* dp = dstates + dst_off(p, bt, c, h) + n;
  float g = 0.0f;
  for (int pp = 0; pp < p.P; ++pp) g += hp[(long)pp * p.N] * dp[(long)pp * p.N];
  g_last[vec_off(p, bt, c, h) + n] = g;
}

template <bool BACK>
static int launch_state_pass(const KP& p, float* states, const float* cs_last, float* dh0_dir, hipStream_t st) {
  const long rows = (long)p.B * p.ndir * p.H * p.P, total = rows * (p.N < 4 ? p.N : (p.N + 3) / 4);
  // Where workgroups of four waves would leave a third of the CUs without one, each wave is one: 2 x 16384 tokens, 8 heads x 32, 256 states,
  // inside a training step, 64 and 67 us -> 55 and 62 (4.6 TB/s, what a copy reaches; 16 or 24 chunks requested ahead: the same); 2 x 1024,
  // forward 7.2 -> 6.7.  With 225 of them, 4 x 1000 tokens, 8 heads x 36, 200 states, 9.5 and 9.2 -> 9.8 and 9.6.
  const int threads = p.N >= 4 && total < 160L * NTHREADS ? 64 : NTHREADS;
  const int blocks = (int)((total + threads - 1) / threads);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads), 0, st, p, states, cs_last, dh0_dir); };
  const bool few = total < (1L << 17) && p.nc >= 16;
  if (p.N < 4) go(&k_state_pass_narrow<BACK>);
  else if (p.N & 3) few ? go(&k_state_pass<8, true, BACK>) : go(&k_state_pass<4, true, BACK>);
  else few ? go(&k_state_pass<8, false, BACK>) : go(&k_state_pass<4, false, BACK>);
  return (int)hipGetLastError();
}

int launch_state_fwd(const KP& p, float* states, const float* cs_last, hipStream_t st) {
  return launch_state_pass<false>(p, states, cs_last, nullptr, st);
}
int launch_state_bwd(const KP& p, const float* cs_last, float* dstates, float* dh0_dir, hipStream_t st) {
  return launch_state_pass<true>(p, dstates, cs_last, dh0_dir, st);
}
int launch_state_sums(const KP& p, const float* states, const float* dstates, float* g_last, hipStream_t st) {
  const long total = (long)p.B * p.ndir * p.nc * p.H * p.N;
  hipLaunchKernelGGL(k_state_sums, dim3((unsigned)((total + NTHREADS - 1) / NTHREADS)), dim3(NTHREADS), 0, st, p, states, dstates, g_last);
  return (int)hipGetLastError();
}

}  // namespace issm
