// C ABI of libissm_hip.so: argument validation, workspace carving and stage sequencing.
// All device work lives in issm_fwd.hip / issm_bwd.hip / rmsnorm_gated.hip.
#include <algorithm>
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "../../include/issm.h"
#include "issm_dev.h"

namespace issm {
int launch_chunk_local(const KP& p, float* states, float* cs_last, float* cabt, bool any, hipStream_t st);
bool bwd_tile_available(const KP& p, const float* dy_ws);
bool bwd_tile_dual(const KP& p, const float* dy_ws, int parts);
int launch_state_fwd(const KP& p, float* states, const float* cs_last, hipStream_t st);
int launch_chunk_scan(const KP& p, const float* states, const float* cabt, float* out_x, hipStream_t st);
int launch_bwd_gate(const KP& p, const float* out_x, float* dy_ws, hipStream_t st);
int launch_bwd_dstates(const KP& p, const float* dy_ws, float* dstates, float* dm, hipStream_t st);
int launch_state_bwd(const KP& p, const float* cs_last, float* dstates, float* dh0_dir, hipStream_t st);
int launch_state_sums(const KP& p, const float* states, const float* dstates, float* g_last, hipStream_t st);
int launch_bwd_chunk(const KP& p, const float* dy_ws, const float* states, const float* dstates, const float* dm,
                     float* partA, float* partBias, int* redo, int* redo_pending, int parts, bool dual, const float* cabt, float* partD,
                     bool* with_dx, hipStream_t st);
int launch_bwd_parts_sum(const KP& p, const int* redo, int parts, hipStream_t st);
int launch_bwd_chunk_redo(const KP& p, int ndirs, const float* dy_ws, const float* states, const float* dstates,
                          const float* dm, float* partA, float* partBias, const int* redo,
                          hipStream_t st);
bool bwd_walk_available(const KP& p, const float* dy_ws);
int launch_bwd_walk(const KP& p, const float* dy_ws, float* dstates, float* dm, float* dh0_dir, hipStream_t st);
int launch_bwd_dx(const KP& p, const float* dy_ws, const float* dstates, const float* cabt, float* partD,
                  hipStream_t st);
int launch_bwd_reduce(const KP& p, const float* partA, const float* partBias, const float* partD,
                      const float* dh0_dir, float* dA, float* dbias, float* dD, float* dh0, hipStream_t st);

int launch_rmsnorm_fwd(const NormP& p, hipStream_t st);
int launch_rmsnorm_bwd(const NormP& p, hipStream_t st);
int launch_hilbert_codes(const HilbertP& p, hipStream_t st);
int launch_hilbert_order(const HilbertOrderP& p, hipStream_t st);
int launch_transpose_states(const TrP& p, hipStream_t st);
int launch_layer_begin(const LayerParamsP& p, const TrP& t, hipStream_t st);
bool layer_behind_takes(const NormP& p);
int launch_layer_behind(const NormP& p, const void* x2, void* sum, const TrP& t, hipStream_t st);
int launch_layer_grads(LayerGradsP& p, const TrP& t, hipStream_t st);
int launch_layer_params(const LayerParamsP& p, hipStream_t st);
bool linear_tile_takes(long tokens, int in, int out, bool nn);
int launch_linear_tile(LinearTileP& p, int njobs, bool nn, hipStream_t st);
int launch_linear(LinearP& p, int njobs, const LayerParamsP* q, hipStream_t st);
int launch_layer_in_tile(LinearTileP& t, LinearP& p, const LayerParamsP& q, hipStream_t st);
int linear_dw_splits(long tokens, int in, int out);
int launch_linear_dw(LinearDwJobs& j, int njobs, hipStream_t st);
int launch_layer_out(LayerOutP& p, hipStream_t st);
int launch_layer_end(LayerOutP& p, LinearP& q, hipStream_t st);
int launch_box_table_bwd(const BoxTableP& p, const float* dtable, void* dw1, void* db1, void* dw2, hipStream_t st);
int launch_box_table(const BoxTableP& p, hipStream_t st);
int launch_fps(int b, int n, int npoint, const float* xyz, float* temp, int* idxs, hipStream_t st);
int launch_ball_query(int b, int n, int m, float radius, int nsample, const float* new_xyz, const float* xyz, int* idx,
                      hipStream_t st);
int launch_group_points(int b, int c, int n, int npoints, int nsample, const float* xyz, const float* centre, float scale,
                        const float* points, const int* idx, float* out, hipStream_t st);
int launch_group_rows_grad(int b, int c, int c0, int cdim, int n, int ms, const float* grad_out, const int* idx,
                           float* grad_points, hipStream_t st);
int launch_interp_rows_grad(int b, int c, int n, int m, const float* grad_out, const int* idx, const float* weight, int* ws,
                            float* grad_points, hipStream_t st);
long interp_rows_grad_ints(int b, int n, int m);
int launch_group_points_grad(int b, int c, int n, int ms, const float* grad_out, const int* idx, float* grad_points,
                             hipStream_t st);
int launch_three_nn(int b, int n, int m, const float* unknown, const float* known, float* dist2, int* idx, hipStream_t st);
int launch_three_interpolate(int b, int c, int m, int n, const float* points, const int* idx, const float* weight, float* out,
                             hipStream_t st);
int launch_three_interpolate_grad(int b, int c, int n, int m, const float* grad_out, const int* idx, const float* weight,
                                  float* grad_points, hipStream_t st);
int launch_scatter_channel_last(bool k3, int b, int c, int n, int ne, const float* grad_out, const int* idx,
                                const float* weight, float* out_cl, hipStream_t st);
int box_dist_workgroups(int B, int L, int K);
int box_dist_bwd_workgroups(int B, int L, int K);
long box_dist_bwd_scratch_bytes(int B, int L, int K, int D, int H, int W);
int launch_box_dist_fwd(const BoxDistP& p, bool only, hipStream_t st);
int launch_box_dist_bwd(const BoxDistP& p, hipStream_t st);
int dwconv_partial_rows(int B, int L, bool chain);
int launch_dwconv_fwd(const DwConvP& p, hipStream_t st);
int launch_conv_pgen(const DwConvP& c, const PGenP& p, hipStream_t st);
int launch_dwconv_bwd(const DwConvP& p, hipStream_t st);
int pgen_bwd_blocks(long tokens);
int launch_pgen_fwd(const PGenP& p, hipStream_t st);
int launch_pgen_bwd(const PGenP& p, hipStream_t st);
}  // namespace issm

using namespace issm;

static thread_local char g_err[512] = "";

static int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

static TensorD td(const issm_tensor& t) {
  TensorD r;
  r.ptr = t.ptr;
  r.s0 = t.stride[0];
  r.s1 = t.stride[1];
  r.s2 = t.stride[2];
  return r;
}

static size_t align64(size_t nfloats) { return (nfloats + 63) & ~(size_t)63; }

struct FwdWs {
  size_t states, cs_last, cabt, out_x, total;  // offsets in floats
};
struct BwdWs {
  size_t dstates, dm, dh0_dir, partA, partBias, partD, redo, dy_ws, ddt_part, dbc_part, total;
};

static int nchunks(const issm_dims& d) { return (d.seqlen + ISSM_CHUNK - 1) / ISSM_CHUNK; }

static FwdWs fwd_layout(const issm_dims& d, bool has_z) {
  const size_t Bt = (size_t)d.batch * d.ndir, nc = nchunks(d), H = d.nheads, P = d.headdim, N = d.dstate;
  FwdWs w;
  size_t o = 0;
  w.states = o; o += align64(Bt * (nc + 1) * H * P * N);
  w.cs_last = o; o += align64(Bt * nc * H * N);
  w.cabt = o; o += align64(Bt * nc * H * ISSM_CHUNK * ISSM_CHUNK);
  w.out_x = o; if (has_z) o += align64(Bt * d.seqlen * H * P);
  w.total = o;
  return w;
}

// How many workgroups of the chunk backward share the heads of a (chunk, group, 64 state columns): as many as fit the 512 places
// of the chip (two workgroups a CU).  A part's sums of dB and dC are 32 KB, which one more launch adds up: 4 us, and as much
// of host time, against 8 us a head and direction; worth it from four of those on (of 4 heads of 2 x 160 tokens, where the host
// sets the pace, it is not).  Where one workgroup each fills the chip, halves only cost that, also where a last round would
// be nearly empty (its workgroups have the CUs to themselves): 9 x 1024 tokens, 8 heads x 32, 256 states, bf16, 576 workgroups,
// a training step 278 us, in halves 281; 320 workgroups, two directions, fp32: 376 and 389.  128 workgroups, 2 x 1024 tokens of
// 8 heads x 36, two directions, bf16: 200 us with one part, 171 - 185, 160 - 169 and 173 with 2, 4 and 8 (three processes each in
// turn; the host sets the pace from two parts on); 64, 1 x 1024 tokens, fp32: 194 and 170 - 184, 158 - 169, 167 - 172.
static int bwd_head_parts(const issm_dims& d) {
  const long blocks = (long)d.batch * nchunks(d) * d.ngroups * ((d.dstate + ISSM_CHUNK - 1) / ISSM_CHUNK);
  const long heads = d.nheads / d.ngroups, most = std::max<long>(1, std::min<long>(heads, 512 / blocks));
  if (d.ndir == 1 && heads % 2 == 0 && blocks <= NCU && most <= 3) return 1;   // (a workgroup takes two heads at a time: bwd_tile_pair)
  const long each = (heads + most - 1) / most;
  return (heads - each) * d.ndir < 4 ? 1 : (int)((heads + each - 1) / each);   // (no part without a head)
}

// Whether the backward's states take one kernel (issm_bwd_walk.hip) or two (k_bwd_dstates, k_state_pass).  Every CU has a walk (256
// of them): one, which saves the states' way through HBM (8 x 4096 tokens, 8 heads x 32, 256 states fp32 174 against 208 us, bf16
// 119 and 152; heads of up to 15, whose walks cost what those of 32 do, go by what follows: 4 x 1536 tokens, 8 heads x 8, 512 states
// 48.5 against 41.2).  Fewer walks wait for latencies one chunk after the other, 3 us and `chunk` for each, while two kernels cost 8 us, 1.3
// more for each 64 columns that k_bwd_dstates loops over, and the chip's share of what the heads and the states of all chunks take.
// Both, us: 2 walks of 64 columns, 4 chunks: heads of 32 9.8 and 11.7 (fp32), 8.7 and 10.6 (bf16), of 64 13.4 and 13.2, 10.8 and 11.6;
// 8 chunks: 16.7 and 12.5, 14.3 and 11.4, 23.6 and 14.0, 18.5 and 12.4.  64 walks of 256 columns, heads of 32, 8 chunks 17.5 and 18.8,
// 15.2 and 16.7; 12 chunks 24.4 and 21.4, 20.9 and 19.2.  192 walks, heads of 64, 8 chunks 29.6 and 32.4; 16 chunks 54.8 and 48.0, bf16 37.9 and
// 40.9.  (Of 5760 sizes the line takes the slower side by more than 8 % in 44, by at most 25 %; a walk for all of up to 8 chunks took
// up to 1.9 times the other side's time.)
static bool bwd_walks(const KP& p, const float* dy) {
  const int heads = p.B * p.ndir * p.H, slices = (p.N + 63) / 64, walks = heads * slices, pt = p.P <= 32 ? 0 : (p.P - 17) / 16;
  static const float chunks_us[2][3] = {{1.35f, 1.55f, 1.9f}, {1.1f, 1.25f, 1.45f}};   // (fp32, bf16; heads of up to 32, 48, 64)
  const float chunk = chunks_us[p.io_dt][pt] + (p.full_tiles ? 0.0f : 0.25f), share = heads * (p.io_dt ? 3e-3f : 4.5e-3f) + (float)walks * p.P * 8e-5f;
  return ((walks >= 256 && p.P >= 16) || p.nc * (chunk - share) <= 4.6f + 1.27f * slices) && bwd_walk_available(p, dy);
}

static bool wants_ddt_part(const issm_scan_args* a) { return a->dims.ndir == 2 && a->dt_dtype == ISSM_BF16; }
// Partial sums that would be rounded to bf16 on their way between kernels: with two directions and a bf16 ddt the first
// direction's share of ddt in fp32 ((B, L, H, N)), with bf16 inputs and incomplete tiles dB and dC of workgroups two
// kernels share (KP::dbc_part).
static BwdWs bwd_layout(const issm_scan_args* a) {
  const issm_dims& d = a->dims;
  const bool has_z = a->z[0].ptr != nullptr, ddt_part = wants_ddt_part(a);
  const size_t Bt = (size_t)d.batch * d.ndir, nc = nchunks(d), H = d.nheads, P = d.headdim, N = d.dstate;
  BwdWs w;
  size_t o = 0;
  w.dstates = o; o += align64(Bt * nc * H * P * N);
  w.dm = o; o += align64(Bt * nc * H * ISSM_CHUNK * ISSM_CHUNK);
  w.dh0_dir = o; o += align64((size_t)d.ndir * d.batch * H * P * N);
  w.partA = o; o += align64(Bt * nc * H * N);
  w.partBias = o; o += align64(Bt * nc * H * N);
  w.partD = o; o += align64(Bt * nc * H * P);
  w.redo = o; o += align64(Bt * nc * H * ((N + ISSM_CHUNK - 1) / ISSM_CHUNK));  // one int per direction, workgroup and head
  w.dy_ws = o; if (has_z) o += align64(Bt * d.seqlen * H * P);
  w.dbc_part = o;
  const int parts = bwd_head_parts(d);
  if (parts > 1) o += Bt * nc * d.ngroups * ((N + ISSM_CHUNK - 1) / ISSM_CHUNK) * parts * 2 * ISSM_CHUNK * ISSM_CHUNK;
  else if (a->io_dtype == ISSM_BF16 && (N % 64 || d.seqlen % ISSM_CHUNK)) o += Bt * nc * d.ngroups * ((N + ISSM_CHUNK - 1) / ISSM_CHUNK) * 2 * ISSM_CHUNK * ISSM_CHUNK;
  w.ddt_part = o; if (ddt_part) o += align64((size_t)d.batch * d.seqlen * H * N);
  w.total = o;
  return w;
}

static int check_dims(const issm_scan_args* a) {
  if (!a) return fail(ISSM_E_NULL, "args is NULL");
  const issm_dims& d = a->dims;
  if (d.batch <= 0 || d.seqlen <= 0 || d.nheads <= 0 || d.headdim <= 0 || d.dstate <= 0 || d.ngroups <= 0)
    return fail(ISSM_E_SHAPE, "non-positive dimension (B=%d L=%d H=%d P=%d N=%d G=%d)", d.batch, d.seqlen, d.nheads,
                d.headdim, d.dstate, d.ngroups);
  if (d.chunk_size <= 0) return fail(ISSM_E_SHAPE, "chunk_size must be positive, got %d", d.chunk_size);
  if (d.nheads % d.ngroups) return fail(ISSM_E_SHAPE, "nheads %d not divisible by ngroups %d", d.nheads, d.ngroups);
  if (d.ndir != 1 && d.ndir != 2) return fail(ISSM_E_SHAPE, "ndir must be 1 or 2, got %d", d.ndir);
  if (d.headdim > MAXP) return fail(ISSM_E_UNSUPPORTED, "headdim %d > %d is not built", d.headdim, MAXP);
  if ((long)d.batch * d.ndir * nchunks(d) * d.nheads > 0x7fffffffL) return fail(ISSM_E_SHAPE, "too many chunk units");
  return ISSM_OK;
}

static int check_strides(const issm_scan_args* a);

static int check_common(const issm_scan_args* a) {
  int rc = check_dims(a);
  if (rc) return rc;
  if ((unsigned)a->io_dtype > 1u || (unsigned)a->dt_dtype > 1u || (unsigned)a->h0_dtype > 1u)
    return fail(ISSM_E_DTYPE, "unknown dtype code (io=%d dt=%d h0=%d)", a->io_dtype, a->dt_dtype, a->h0_dtype);
  if (a->flags & ISSM_FLAG_SEQ_IDX) {
    if (!a->seq_idx) return fail(ISSM_E_NULL, "ISSM_FLAG_SEQ_IDX is set and seq_idx is NULL");
    if (a->dims.ndir != 1) return fail(ISSM_E_UNSUPPORTED, "seq_idx with ndir = %d (one direction only)", a->dims.ndir);
    if (a->seq_idx_stride[0] < 0 || a->seq_idx_stride[1] < 0 ||
        a->seq_idx_stride[1] * (int64_t)a->dims.seqlen >= ((int64_t)1 << 31))
      return fail(ISSM_E_STRIDE, "seq_idx strides (%lld, %lld)", (long long)a->seq_idx_stride[0], (long long)a->seq_idx_stride[1]);
  }
  if (!(a->dt_min >= 0.0f)) return fail(ISSM_E_UNSUPPORTED, "dt_limit[0] = %g < 0 is not supported", a->dt_min);
  if (!(a->dt_max >= a->dt_min)) return fail(ISSM_E_SHAPE, "dt_limit is empty (%g, %g)", a->dt_min, a->dt_max);
  if (!a->A) return fail(ISSM_E_NULL, "A is NULL");
  if (!a->dt.ptr) return fail(ISSM_E_NULL, "dt is NULL");
  for (int dir = 0; dir < a->dims.ndir; ++dir) {
    if (!a->x[dir].ptr || !a->Bm[dir].ptr || !a->Cm[dir].ptr)
      return fail(ISSM_E_NULL, "x/B/C of direction %d is NULL", dir);
    if ((a->z[0].ptr != nullptr) != (a->z[dir].ptr != nullptr))
      return fail(ISSM_E_NULL, "z must be given for all directions or none");
  }
  return check_strides(a);
}

// The kernels address a row of a caller tensor as a 64-bit (batch, head) base plus a 32-bit BYTE
// offset (time row * stride[1] + column) * element size: that offset must fit (2^30 elements), and
// strides may not be negative.
static int check_td(const issm_tensor& t, const char* name, int dir, long rows, long inner) {
  if (!t.ptr) return ISSM_OK;
  for (int i = 0; i < 3; ++i)
    if (t.stride[i] < 0) return fail(ISSM_E_STRIDE, "%s[%d]: negative stride %ld", name, dir, (long)t.stride[i]);
  if ((rows - 1) * (long)t.stride[1] + inner > 0x3fffffffL)
    return fail(ISSM_E_STRIDE, "%s[%d]: seqlen * stride[1] = %ld * %ld exceeds the 32-bit row offset range", name, dir,
                rows, (long)t.stride[1]);
  return ISSM_OK;
}

static int check_strides(const issm_scan_args* a) {
  const issm_dims& d = a->dims;
  int rc;
  for (int i = 0; i < d.ndir; ++i) {
    if ((rc = check_td(a->x[i], "x", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->z[i], "z", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->out[i], "out", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->dout[i], "dout", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->dx[i], "dx", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->dz[i], "dz", i, d.seqlen, d.headdim))) return rc;
    if ((rc = check_td(a->Bm[i], "B", i, d.seqlen, d.dstate))) return rc;
    if ((rc = check_td(a->Cm[i], "C", i, d.seqlen, d.dstate))) return rc;
    if ((rc = check_td(a->dB[i], "dB", i, d.seqlen, d.dstate))) return rc;
    if ((rc = check_td(a->dC[i], "dC", i, d.seqlen, d.dstate))) return rc;
  }
  if ((rc = check_td(a->dt, "dt", 0, d.seqlen, d.dstate))) return rc;
  if ((rc = check_td(a->ddt, "ddt", 0, d.seqlen, d.dstate))) return rc;
  if ((rc = check_td(a->h0, "initial_states", 0, d.nheads, d.dstate))) return rc;
  return ISSM_OK;
}

static KP make_kp(const issm_scan_args* a) {
  KP p;
  memset(&p, 0, sizeof(p));
  const issm_dims& d = a->dims;
  p.B = d.batch; p.L = d.seqlen; p.H = d.nheads; p.P = d.headdim; p.N = d.dstate; p.G = d.ngroups;
  p.ndir = d.ndir; p.nc = nchunks(d); p.hpg = d.nheads / d.ngroups; p.dir0 = 0;
  p.io_dt = a->io_dtype; p.dt_dt = a->dt_dtype; p.h0_dt = a->h0_dtype;
  p.flags = ((a->flags & ISSM_FLAG_DT_SOFTPLUS) ? F_SOFTPLUS : 0u) | ((a->flags & ISSM_FLAG_D_HAS_HDIM) ? F_D_HDIM : 0u);
  p.dt_min = a->dt_min; p.dt_max = a->dt_max;
  // softplus is positive: limits of (<= 0, >= 3e38 or inf) cannot act on it
  if ((p.flags & F_SOFTPLUS) && a->dt_min <= 0.0f && a->dt_max >= 3.0e38f) p.flags |= F_NOCLAMP;
  for (int i = 0; i < 2; ++i) {
    p.x[i] = td(a->x[i]); p.Bm[i] = td(a->Bm[i]); p.Cm[i] = td(a->Cm[i]); p.z[i] = td(a->z[i]);
    p.out[i] = td(a->out[i]); p.dout[i] = td(a->dout[i]); p.dx[i] = td(a->dx[i]); p.dB[i] = td(a->dB[i]);
    p.dC[i] = td(a->dC[i]); p.dz[i] = td(a->dz[i]);
    p.final_states[i] = a->final_states[i];
    p.dfinal[i] = a->dfinal[i];
  }
  p.dt = td(a->dt); p.ddt = td(a->ddt); p.h0 = td(a->h0);
  p.A = a->A; p.D = a->D; p.dt_bias = a->dt_bias;
  if (a->flags & ISSM_FLAG_SEQ_IDX) {
    p.seq_idx = a->seq_idx; p.seq_s0 = a->seq_idx_stride[0]; p.seq_s1 = a->seq_idx_stride[1];
  }
  p.by_H = div_by(p.H); p.by_nc = div_by(p.nc); p.by_hpg = div_by(p.hpg); p.by_slices = div_by((p.N + NS - 1) / NS); p.by_G = div_by(p.G);
  p.by_quads = div_by((p.N + 3) / 4); p.by_P = div_by(p.P);
  p.full_tiles = p.N % 64 == 0 && p.L % ISSM_CHUNK == 0 && !p.seq_idx;
  return p;
}

static int launched(int hip_err, const char* what) {
  if (hip_err == 0) return ISSM_OK;
  return fail(ISSM_E_LAUNCH, "%s: %s", what, hipGetErrorString((hipError_t)hip_err));
}

static void norm_scratch_warm(hipStream_t stream);  // further down, with the allocation-free backward it serves

extern "C" {

int issm_abi_version(void) { return ISSM_ABI_VERSION; }
const char* issm_last_error(void) { return g_err; }

int issm_fwd_workspace_bytes(const issm_scan_args* a, size_t* out) {
  int rc = check_dims(a);
  if (rc) return rc;
  if (!out) return fail(ISSM_E_NULL, "out is NULL");
  *out = fwd_layout(a->dims, a->z[0].ptr != nullptr).total * sizeof(float);
  return ISSM_OK;
}

int issm_bwd_workspace_bytes(const issm_scan_args* a, size_t* out) {
  int rc = check_dims(a);
  if (rc) return rc;
  if (!out) return fail(ISSM_E_NULL, "out is NULL");
  *out = bwd_layout(a).total * sizeof(float);
  return ISSM_OK;
}

int issm_stage_chunk_local(const issm_scan_args* a, float* states, float* cs_last, float* cabt) {
  int rc = check_common(a);
  if (rc) return rc;
  if (!cs_last) return fail(ISSM_E_NULL, "cs_last is NULL");
  KP p = make_kp(a);
  return launched(launch_chunk_local(p, states, cs_last, cabt, false, (hipStream_t)a->stream), "chunk_local");
}

int issm_stage_state_passing_fwd(const issm_scan_args* a, float* states, const float* cs_last) {
  int rc = check_dims(a);
  if (rc) return rc;
  if (!states || !cs_last) return fail(ISSM_E_NULL, "states/cs_last is NULL");
  KP p = make_kp(a);
  return launched(launch_state_fwd(p, states, cs_last, (hipStream_t)a->stream), "state_passing_fwd");
}

int issm_stage_chunk_scan(const issm_scan_args* a, const float* states, const float* cabt, float* out_x) {
  int rc = check_common(a);
  if (rc) return rc;
  if (!states || !cabt) return fail(ISSM_E_NULL, "states/cabt is NULL");
  for (int dir = 0; dir < a->dims.ndir; ++dir)
    if (!a->out[dir].ptr) return fail(ISSM_E_NULL, "out of direction %d is NULL", dir);
  if (a->z[0].ptr && !out_x) return fail(ISSM_E_NULL, "out_x is required when z is given");
  KP p = make_kp(a);
  return launched(launch_chunk_scan(p, states, cabt, out_x, (hipStream_t)a->stream), "chunk_scan");
}

static int scan_fwd(const issm_scan_args* a, bool forward_only) {
  int rc = check_common(a);
  if (rc) return rc;
  const bool has_z = a->z[0].ptr != nullptr;
  const FwdWs w = fwd_layout(a->dims, has_z);
  if (!a->workspace || a->workspace_bytes < w.total * sizeof(float))
    return fail(ISSM_E_WORKSPACE, "forward workspace: need %zu bytes, got %zu", w.total * sizeof(float),
                a->workspace ? a->workspace_bytes : (size_t)0);
  for (int dir = 0; dir < a->dims.ndir; ++dir)
    if (!a->out[dir].ptr) return fail(ISSM_E_NULL, "out of direction %d is NULL", dir);
  float* ws = (float*)a->workspace;
  KP p = make_kp(a);
  hipStream_t st = (hipStream_t)a->stream;
  if ((rc = launched(launch_chunk_local(p, ws + w.states, ws + w.cs_last, ws + w.cabt, forward_only, st), "chunk_local"))) return rc;
  if ((rc = launched(launch_state_fwd(p, ws + w.states, ws + w.cs_last, st), "state_passing_fwd"))) return rc;
  return launched(launch_chunk_scan(p, ws + w.states, ws + w.cabt, has_z ? ws + w.out_x : nullptr, st), "chunk_scan");
}

int issm_scan_fwd(const issm_scan_args* a) { return scan_fwd(a, false); }
int issm_scan_fwd_only(const issm_scan_args* a) { return scan_fwd(a, true); }

int issm_stage_bwd_gate(const issm_scan_args* a, const float* out_x, float* dy_gated) {
  int rc = check_common(a);
  if (rc) return rc;
  if (!out_x || !dy_gated || !a->z[0].ptr) return fail(ISSM_E_NULL, "out_x/dy_gated/z is NULL");
  KP p = make_kp(a);
  return launched(launch_bwd_gate(p, out_x, dy_gated, (hipStream_t)a->stream), "bwd_gate");
}

static int check_dout(const issm_scan_args* a, const float* dy_gated) {
  if (dy_gated) return ISSM_OK;
  for (int dir = 0; dir < a->dims.ndir; ++dir)
    if (!a->dout[dir].ptr) return fail(ISSM_E_NULL, "dout of direction %d is NULL", dir);
  return ISSM_OK;
}

int issm_stage_bwd_dstates(const issm_scan_args* a, const float* dy_gated, float* dstates, float* dm) {
  int rc = check_common(a);
  if (rc) return rc;
  if ((rc = check_dout(a, dy_gated))) return rc;
  KP p = make_kp(a);
  return launched(launch_bwd_dstates(p, dy_gated, dstates, dm, (hipStream_t)a->stream), "bwd_dstates");
}

int issm_stage_state_passing_bwd(const issm_scan_args* a, const float* states, const float* cs_last, float* dstates,
                                 float* g_last, float* dh0_dir) {
  int rc = check_dims(a);
  if (rc) return rc;
  if (!cs_last || !dstates || !dh0_dir || (g_last && !states)) return fail(ISSM_E_NULL, "state_passing_bwd: NULL buffer");
  KP p = make_kp(a);
  hipStream_t st = (hipStream_t)a->stream;
  if ((rc = launched(launch_state_bwd(p, cs_last, dstates, dh0_dir, st), "state_passing_bwd")) || !g_last) return rc;
  return launched(launch_state_sums(p, states, dstates, g_last, st), "state_passing_bwd (sums)");
}

int issm_stage_bwd_states(const issm_scan_args* a, const float* dy_gated, const float* states, float* dstates, float* dm,
                          float* g_last, float* dh0_dir) {
  int rc = check_common(a);
  if (rc) return rc;
  if ((rc = check_dout(a, dy_gated))) return rc;
  if (!dstates || !dm || !dh0_dir || (g_last && !states)) return fail(ISSM_E_NULL, "bwd_states: NULL buffer");
  KP p = make_kp(a);
  if (!bwd_walk_available(p, dy_gated)) return fail(ISSM_E_UNSUPPORTED, "bwd_states: packed sequences, mixed types, or rows of x or dy that are no multiple of four elements");
  hipStream_t st = (hipStream_t)a->stream;
  if ((rc = launched(launch_bwd_walk(p, dy_gated, dstates, dm, dh0_dir, st), "bwd_states")) || !g_last) return rc;
  return launched(launch_state_sums(p, states, dstates, g_last, st), "bwd_states (sums)");
}

size_t issm_bwd_chunk_redo_ints(const issm_scan_args* a) {
  if (check_dims(a)) return 0;
  const issm_dims& d = a->dims;
  return (size_t)d.batch * d.ndir * nchunks(d) * d.nheads * ((d.dstate + ISSM_CHUNK - 1) / ISSM_CHUNK);
}

int issm_stage_bwd_chunk(const issm_scan_args* a, int dir, const float* dy_gated, const float* states,
                         const float* dstates, const float* dm, const float* /*g_last*/, float* part_a,
                         float* part_bias, int32_t* redo) {
  int rc = check_common(a);
  if (rc) return rc;
  if ((rc = check_dout(a, dy_gated))) return rc;
  if (dir < -1 || dir >= a->dims.ndir) return fail(ISSM_E_SHAPE, "dir %d out of range", dir);
  if (!states || !dstates || !dm || !part_a || !part_bias) return fail(ISSM_E_NULL, "bwd_chunk: NULL buffer");
  KP p = make_kp(a);
  hipStream_t st = (hipStream_t)a->stream;
  const bool dual = dir < 0 && redo && bwd_tile_dual(p, dy_gated, bwd_head_parts(a->dims));
  const int first = std::max(dir, 0), last = dir < 0 && !dual ? p.ndir - 1 : first;
  int pending = 0;
  for (int d = first; d <= last; ++d) {
    p.dir0 = d;
    if ((rc = launched(launch_bwd_chunk(p, dy_gated, states, dstates, dm, part_a, part_bias, redo, &pending, 1, dual,
                                        nullptr, nullptr, nullptr, st),
                       "bwd_chunk")))
      return rc;
    if (pending && (rc = launched(launch_bwd_chunk_redo(p, dual ? 2 : 1, dy_gated, states, dstates, dm, part_a, part_bias, redo, st),
                                  "bwd_chunk (redo)")))
      return rc;
  }
  return ISSM_OK;
}

int issm_stage_bwd_dx(const issm_scan_args* a, const float* dy_gated, const float* dstates, const float* cabt,
                      float* part_d) {
  int rc = check_common(a);
  if (rc) return rc;
  if ((rc = check_dout(a, dy_gated))) return rc;
  if (!dstates || !cabt) return fail(ISSM_E_NULL, "bwd_dx: NULL buffer");
  if (a->D && a->dD && !part_d) return fail(ISSM_E_NULL, "bwd_dx: part_d is NULL");
  KP p = make_kp(a);
  return launched(launch_bwd_dx(p, dy_gated, dstates, cabt, part_d, (hipStream_t)a->stream), "bwd_dx");
}

int issm_stage_bwd_reduce(const issm_scan_args* a, const float* part_a, const float* part_bias, const float* part_d,
                          const float* dh0_dir) {
  int rc = check_dims(a);
  if (rc) return rc;
  KP p = make_kp(a);
  return launched(launch_bwd_reduce(p, part_a, part_bias, part_d, dh0_dir, part_a ? a->dA : nullptr,
                                    (part_bias && a->dt_bias) ? a->ddt_bias : nullptr,
                                    (part_d && a->D) ? a->dD : nullptr, dh0_dir ? a->dh0 : nullptr,
                                    (hipStream_t)a->stream),
                  "bwd_reduce");
}

int issm_bwd_walks(const issm_scan_args* a) {
  if (check_common(a)) return 0;
  const KP p = make_kp(a);
  // a gated dy is the workspace's; whatever its address, its rows are whole
  return bwd_walks(p, a->z[0].ptr ? reinterpret_cast<const float*>(a->z[0].ptr) : nullptr) ? 1 : 0;
}

int issm_scan_bwd(const issm_scan_args* a) {
  int rc = check_common(a);
  if (rc) return rc;
  const bool has_z = a->z[0].ptr != nullptr;
  const FwdWs fw = fwd_layout(a->dims, has_z);
  const BwdWs bw = bwd_layout(a);
  if (!a->saved) return fail(ISSM_E_WORKSPACE, "saved forward workspace is NULL");
  if (!a->bwd_workspace || a->bwd_workspace_bytes < bw.total * sizeof(float))
    return fail(ISSM_E_WORKSPACE, "backward workspace: need %zu bytes, got %zu", bw.total * sizeof(float),
                a->bwd_workspace ? a->bwd_workspace_bytes : (size_t)0);
  for (int dir = 0; dir < a->dims.ndir; ++dir)
    if (!a->dout[dir].ptr) return fail(ISSM_E_NULL, "dout of direction %d is NULL", dir);
  const float* sv = (const float*)a->saved;
  float* ws = (float*)a->bwd_workspace;
  KP p = make_kp(a);
  hipStream_t st = (hipStream_t)a->stream;
  const float* dy = nullptr;
  if (has_z) {
    if ((rc = launched(launch_bwd_gate(p, sv + fw.out_x, ws + bw.dy_ws, st), "bwd_gate"))) return rc;
    dy = ws + bw.dy_ws;
  }
  if (bwd_walks(p, dy)) {
    if ((rc = launched(launch_bwd_walk(p, dy, ws + bw.dstates, ws + bw.dm, ws + bw.dh0_dir, st), "bwd_states"))) return rc;
  } else {
    if ((rc = launched(launch_bwd_dstates(p, dy, ws + bw.dstates, ws + bw.dm, st), "bwd_dstates"))) return rc;
    if ((rc = launched(launch_state_bwd(p, sv + fw.cs_last, ws + bw.dstates, ws + bw.dh0_dir, st), "state_passing_bwd"))) return rc;
  }
  int* redo = reinterpret_cast<int*>(ws + bw.redo);
  int pending = 0;
  KP pc = p;
  int parts = 1;
  if (bwd_tile_available(p, dy)) {
    parts = bwd_head_parts(a->dims);
    if (parts > 1 || (p.io_dt && !p.full_tiles)) p.dbc_part = pc.dbc_part = ws + bw.dbc_part;
  }
  const bool dual = bwd_tile_dual(p, dy, parts);
  bool with_dx = false;   // the chunk backward's launch has dx
  if (wants_ddt_part(a) && !dual && bwd_tile_available(p, dy)) {
    // both directions go through the tile-base kernel: the first one's share of the bf16 ddt travels in fp32
    pc.ddt_part.ptr = ws + bw.ddt_part;
    pc.ddt_part.s2 = p.N;
    pc.ddt_part.s1 = (long)p.H * p.N;
    pc.ddt_part.s0 = (long)p.L * p.H * p.N;
  }
  for (int dir = 0; dir < (dual ? 1 : p.ndir); ++dir) {
    KP pd = pc;
    pd.dir0 = dir;
    if ((rc = launched(launch_bwd_chunk(pd, dy, sv + fw.states, ws + bw.dstates, ws + bw.dm,
                                        ws + bw.partA, ws + bw.partBias, redo, &pending, parts, dual, sv + fw.cabt, ws + bw.partD, &with_dx, st),
                       "bwd_chunk")))
      return rc;
  }
  if (parts > 1 && (rc = launched(launch_bwd_parts_sum(p, redo, parts, st), "bwd_chunk (parts)"))) return rc;
  const int together = p.L % ISSM_CHUNK == 0 ? p.ndir : 1;   // directions per launch of the pass over the marks
  for (int dir = 0; pending && dir < p.ndir; dir += together) {
    KP pd = p;
    pd.dir0 = dir;
    if ((rc = launched(launch_bwd_chunk_redo(pd, together, dy, sv + fw.states, ws + bw.dstates, ws + bw.dm,
                                             ws + bw.partA, ws + bw.partBias, redo, st),
                       "bwd_chunk (redo)")))
      return rc;
  }
  if (!with_dx && (rc = launched(launch_bwd_dx(p, dy, ws + bw.dstates, sv + fw.cabt, ws + bw.partD, st), "bwd_dx"))) return rc;
  return launched(launch_bwd_reduce(p, ws + bw.partA, ws + bw.partBias, ws + bw.partD, ws + bw.dh0_dir, a->dA,
                                    a->dt_bias ? a->ddt_bias : nullptr, a->D ? a->dD : nullptr, a->dh0, st),
                  "bwd_reduce");
}

// ------------------------------------------------------------------ gated RMSNorm
int issm_rmsnorm_bwd_blocks(int64_t rows) {
  if (rows <= 0) return 0;
  return (int)(rows < 2048 ? rows : 2048);
}

static int norm_params(const issm_norm_args* a, NormP* p, bool bwd, bool part = false) {
  if (!a) return fail(ISSM_E_NULL, "args is NULL");
  if (a->rows <= 0 || a->ncols <= 0) return fail(ISSM_E_SHAPE, "rmsnorm: rows=%lld ncols=%d", (long long)a->rows, a->ncols);
  const int gs = a->group_size > 0 ? a->group_size : a->ncols;
  if (a->ncols % gs) return fail(ISSM_E_SHAPE, "rmsnorm: ncols %d not divisible by group_size %d", a->ncols, gs);
  if ((unsigned)a->dtype > 1u || (unsigned)a->weight_dtype > 1u) return fail(ISSM_E_DTYPE, "rmsnorm: unknown dtype");
  if (!a->x || !a->w || !a->rstd) return fail(ISSM_E_NULL, "rmsnorm: x/w/rstd is NULL");
  if (a->ncols > 16384) return fail(ISSM_E_UNSUPPORTED, "rmsnorm: ncols %d > 16384", a->ncols);
  if (!bwd && !a->y) return fail(ISSM_E_NULL, "rmsnorm: y is NULL");
  if (bwd && (!a->dy || !a->dx || !a->dw_partial || (!a->dw && !part))) return fail(ISSM_E_NULL, "rmsnorm bwd: NULL buffer");
  if (bwd && a->z && !a->dz) return fail(ISSM_E_NULL, "rmsnorm bwd: dz is NULL");
  if (a->layer_norm && !a->mean) return fail(ISSM_E_NULL, "layernorm: mean is NULL");
  if (bwd && a->bias && (!a->db_partial || !a->db)) return fail(ISSM_E_NULL, "norm bwd with bias: db_partial/db is NULL");
  // only the backward stages the bias partial sums next to the weight's in LDS; the forward has no such limit
  if (bwd && a->bias && a->ncols > 8192 && !(a->ncols / gs == 1 && (a->ncols & 3) == 0 && a->ncols <= 1024))
    return fail(ISSM_E_UNSUPPORTED, "norm bwd with bias: ncols %d > 8192", a->ncols);
  p->rows = a->rows; p->ncols = a->ncols; p->gs = gs; p->ngroups = a->ncols / gs;
  p->dt = a->dtype; p->wdt = a->weight_dtype; p->nbg = a->norm_before_gate; p->eps = a->eps;
  p->x = a->x; p->z = a->z; p->w = a->w; p->xs = a->x_row_stride; p->zs = a->z_row_stride;
  p->y = a->y; p->ys = a->y_row_stride; p->rstd = a->rstd;
  p->dy = a->dy; p->dys = a->dy_row_stride; p->dx = a->dx; p->dz = a->dz; p->dxs = a->dx_row_stride;
  p->dzs = a->dz_row_stride; p->dw_partial = a->dw_partial; p->dw = a->dw; p->dw_dt = ISSM_F32;
  p->nblocks = issm_rmsnorm_bwd_blocks(a->rows);
  p->ln = a->layer_norm ? 1 : 0; p->b = a->bias; p->mean = a->mean; p->db_partial = a->db_partial; p->db = a->db;
  return ISSM_OK;
}

int issm_gated_rmsnorm_fwd(const issm_norm_args* a) {
  NormP p;
  int rc = norm_params(a, &p, false);
  if (rc) return rc;
  norm_scratch_warm((hipStream_t)a->stream);
  return launched(launch_rmsnorm_fwd(p, (hipStream_t)a->stream), "rmsnorm_fwd");
}

int issm_gated_rmsnorm_bwd(const issm_norm_args* a) {
  NormP p;
  int rc = norm_params(a, &p, true);
  if (rc) return rc;
  norm_scratch_warm((hipStream_t)a->stream);
  return launched(launch_rmsnorm_bwd(p, (hipStream_t)a->stream), "rmsnorm_bwd");
}

int issm_gated_rmsnorm_bwd_as(const issm_norm_args* a, int32_t grad_dtype) {
  NormP p;
  int rc = norm_params(a, &p, true);
  if (rc) return rc;
  if ((unsigned)grad_dtype > 1u) return fail(ISSM_E_DTYPE, "rmsnorm: unknown dtype");
  norm_scratch_warm((hipStream_t)a->stream);
  p.dw_dt = grad_dtype;
  return launched(launch_rmsnorm_bwd(p, (hipStream_t)a->stream), "rmsnorm_bwd_as");
}

int issm_gated_rmsnorm_bwd_part(const issm_norm_args* a) {
  NormP p;
  int rc = norm_params(a, &p, true, true);
  if (rc) return rc;
  if (p.b) return fail(ISSM_E_UNSUPPORTED, "rmsnorm_bwd_part: no bias");
  norm_scratch_warm((hipStream_t)a->stream);
  p.dw = nullptr;
  return launched(launch_rmsnorm_bwd(p, (hipStream_t)a->stream), "rmsnorm_bwd_part");
}

}  // extern "C"

// ---- the same backward on a scratch buffer that belongs to the library: no allocation by anyone
// The per-block partial sums of dw (nblocks x ncols floats) normally arrive as args->dw_partial.  For callers that
// cannot allocate, they go into this array instead; every GPU the library runs on holds its own copy (8 MiB) at
// its own address until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress: the device address is looked up once per device and kept, and it is that pointer -- never
// the name -- that the kernels receive.  (No `used` attribute on the array: the compiler gives a file-scope device
// variable that host code refers to an external symbol, which is what the runtime's lookup needs; `used` keeps it local
// and the lookup then aborts the process.)
static __device__ __align__(256) float g_norm_scratch[ISSM_NORM_SCRATCH_FLOATS];
static constexpr int kMaxDevices = 64;
static std::mutex g_norm_scratch_mutex;
static float* g_norm_scratch_ptr[kMaxDevices];  // [device]: address of that device's copy, once looked up
static std::atomic<bool> g_norm_scratch_known[kMaxDevices];  // set after the pointer: a cheap test for norm_scratch_warm

// The look-up may load the code object and so must not run while `stream` records a graph: a first call on a device
// that arrives under capture is refused (one eager call per device, of this entry point or of any other of the
// library's normalisation calls, comes first -- those resolve the address on the way, see norm_scratch_warm).
static int norm_scratch_ptr(float** out, hipStream_t stream) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(ISSM_E_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(ISSM_E_UNSUPPORTED, "device index %d outside 0..%d", dev, kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(g_norm_scratch_mutex);
  if (!g_norm_scratch_ptr[dev]) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone)
      return fail(ISSM_E_UNSUPPORTED,
                  "rmsnorm bwd without allocation: the first call on device %d came while its stream records a graph; "
                  "make one eager call of a normalisation entry point on this device before the capture", dev);
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_norm_scratch));  // of the current device's copy
    if (e != hipSuccess || !ptr)
      return fail(ISSM_E_LAUNCH, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_norm_scratch_ptr[dev] = (float*)ptr;
    g_norm_scratch_known[dev].store(true, std::memory_order_release);
  }
  *out = g_norm_scratch_ptr[dev];
  return ISSM_OK;
}
// Called by the other normalisation entry points: resolves the current device's address when that is possible now
// (not under capture), silently otherwise, so that a model whose forward ran eagerly once can capture the
// allocation-free backward without a warm-up call of its own.
static void norm_scratch_warm(hipStream_t stream) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return;
  }
  if (g_norm_scratch_known[dev].load(std::memory_order_acquire)) return;
  float* unused = nullptr;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return;
  }
  if (norm_scratch_ptr(&unused, stream) != ISSM_OK) g_err[0] = 0;
}

extern "C" {

int issm_gated_rmsnorm_bwd_noalloc(const issm_norm_args* a) {
  if (!a) return fail(ISSM_E_NULL, "args is NULL");
  issm_norm_args b = *a;
  float* scratch = nullptr;
  // sizes are checked before anything touches the device
  const int64_t part = b.rows > 0 && b.ncols > 0 ? (int64_t)issm_rmsnorm_bwd_blocks(b.rows) * b.ncols : 0;
  const int64_t need = part * (b.bias ? 2 : 1);  // the partial sums of dw, then those of db
  if (need > (int64_t)ISSM_NORM_SCRATCH_FLOATS)
    return fail(ISSM_E_WORKSPACE,
                "rmsnorm bwd without allocation: %d row blocks x %d columns%s = %lld floats of partial sums exceed the "
                "library's %d-float scratch array; use issm_gated_rmsnorm_bwd with a dw_partial buffer",
                issm_rmsnorm_bwd_blocks(b.rows), b.ncols, b.bias ? " x 2 (weight and bias)" : "", (long long)need,
                (int)ISSM_NORM_SCRATCH_FLOATS);
  // placeholders so that the shared validation sees buffers; replaced below
  b.dw_partial = (float*)(uintptr_t)256;
  b.db_partial = (float*)(uintptr_t)256;
  NormP p;
  int rc = norm_params(&b, &p, true);
  if (rc) return rc;
  if ((rc = norm_scratch_ptr(&scratch, (hipStream_t)a->stream))) return rc;
  p.dw_partial = scratch;  // every launched block writes its whole row of partials before the sum reads it
  p.db_partial = scratch + part;
  return launched(launch_rmsnorm_bwd(p, (hipStream_t)a->stream), "rmsnorm_bwd_noalloc");
}

static int pgen_params(const issm_pgen_args* a, PGenP* p, bool bwd, bool forward_only = false, bool conv = false, bool part = false) {
  if (!a) return fail(ISSM_E_NULL, "param_gen: args is NULL");
  if (a->tokens < 0 || a->K < 0 || a->H < 1 || a->G < 1) return fail(ISSM_E_SHAPE, "param_gen: bad shape");
  if (a->M != 16) return fail(ISSM_E_UNSUPPORTED, "param_gen: M = %d (only 16 is built)", a->M);
  if (a->H + 2 * a->G > 12) return fail(ISSM_E_UNSUPPORTED, "param_gen: H + 2G = %d > 12", a->H + 2 * a->G);
  if (a->dtype != ISSM_F32 && a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "param_gen: dtype %d", a->dtype);
  if (a->tokens * (int64_t)a->K * 16 >= ((int64_t)1 << 40)) return fail(ISSM_E_SHAPE, "param_gen: too large");
  if (!a->dist || !a->W) return fail(ISSM_E_NULL, "param_gen: dist/W is NULL");
  if (a->weights && !a->dt_raw && !forward_only) return fail(ISSM_E_NULL, "param_gen: weights given but dt_raw is NULL");
  if (!bwd) {
    if (!a->dt || !a->Bm || !a->Cm) return fail(ISSM_E_NULL, "param_gen: dt/Bm/Cm is NULL");
    if (!a->bias && (!a->tok || !a->tok_add || (!a->tail && !conv))) return fail(ISSM_E_NULL, "param_gen: neither bias nor tok/tok_add/tail");
    if (!a->bias && a->tok_stride < a->H) return fail(ISSM_E_STRIDE, "param_gen: tok_stride %lld", (long long)a->tok_stride);
    if (a->has_back && (!a->Bm_back || !a->Cm_back)) return fail(ISSM_E_NULL, "param_gen: Bm_back/Cm_back is NULL");
  } else {
    if (!a->dw_partial || (!a->dW && !part)) return fail(ISSM_E_NULL, "param_gen bwd: dw_partial/dW is NULL");
  }
  p->tokens = a->tokens; p->K = a->K; p->H = a->H; p->G = a->G; p->dtype = a->dtype; p->has_back = a->has_back ? 1 : 0;
  p->dist = a->dist; p->W = a->W; p->bias = a->bias;
  p->tok = a->tok; p->tok_stride = a->tok_stride; p->tok_add = a->tok_add; p->tail = a->tail;
  p->dt = a->dt; p->Bm = a->Bm; p->Cm = a->Cm; p->Bb = a->Bm_back; p->Cb = a->Cm_back;
  p->ddt = a->ddt; p->dB = a->dBm; p->dC = a->dCm; p->dBb = a->dBm_back; p->dCb = a->dCm_back;
  p->weights = a->weights; p->dt_raw = a->dt_raw; p->dweights = a->weights ? a->dweights : nullptr;
  if (a->dbias_sum && !a->dbias) return fail(ISSM_E_NULL, "param_gen: dbias_sum needs dbias");
  p->dbias_sum = a->dbias_sum;
  p->ddist = a->ddist; p->dbias = a->dbias; p->dw_partial = a->dw_partial; p->dW = a->dW;
  p->nblocks = pgen_bwd_blocks(a->tokens);
  p->dtok = p->dtail = nullptr;
  p->dtok_stride = 0;
  p->bias_partial = nullptr;
  return ISSM_OK;
}

int issm_param_gen_bwd_blocks(int64_t tokens) { return tokens > 0 ? pgen_bwd_blocks(tokens) : 0; }

int issm_param_gen_fwd(const issm_pgen_args* a) {
  PGenP p;
  int rc = pgen_params(a, &p, false);
  if (rc) return rc;
  if (p.tokens == 0 || p.K == 0) return ISSM_OK;
  return launched(launch_pgen_fwd(p, (hipStream_t)a->stream), "param_gen_fwd");
}

int issm_param_gen_fwd_only(const issm_pgen_args* a) {
  PGenP p;
  int rc = pgen_params(a, &p, false, true);
  if (rc) return rc;
  if (p.tokens == 0 || p.K == 0) return ISSM_OK;
  p.dt_raw = nullptr;
  return launched(launch_pgen_fwd(p, (hipStream_t)a->stream), "param_gen_fwd_only");
}

int issm_param_gen_bwd(const issm_pgen_args* a) {
  PGenP p;
  int rc = pgen_params(a, &p, true);
  if (rc) return rc;
  if (p.tokens == 0) return ISSM_OK;
  return launched(launch_pgen_bwd(p, (hipStream_t)a->stream), "param_gen_bwd");
}

int issm_param_gen_bwd_part(const issm_pgen_args* a, const issm_pgen_producers* b) {
  PGenP p;
  int rc = pgen_params(a, &p, true, false, false, true);
  if (rc) return rc;
  if (!b || !b->dtok || !b->dtail || !a->has_back) return fail(ISSM_E_NULL, "param_gen bwd: dtok/dtail is NULL, or has_back is 0");
  if (b->dtok_stride < a->H) return fail(ISSM_E_STRIDE, "param_gen bwd: dtok_stride %lld", (long long)b->dtok_stride);
  if (p.tokens == 0) return ISSM_OK;
  p.dW = p.dbias_sum = nullptr;
  p.dtok = b->dtok; p.dtok_stride = b->dtok_stride; p.dtail = b->dtail;
  p.bias_partial = p.dw_partial + (long)p.nblocks * (p.H + 2 * p.G) * 16;
  return launched(launch_pgen_bwd(p, (hipStream_t)a->stream), "param_gen_bwd_part");
}

static int dwconv_params(const issm_dwconv_args* a, DwConvP* p, bool bwd, bool heads_only = false, bool part = false) {
  if (!a) return fail(ISSM_E_NULL, "dwconv: args is NULL");
  if (a->batch < 0 || a->seqlen < 0 || a->channels < 1) return fail(ISSM_E_SHAPE, "dwconv: bad shape");
  if (a->taps != 7) return fail(ISSM_E_UNSUPPORTED, "dwconv: %d taps (only 7 is built)", a->taps);
  if (a->nsets < 1 || a->nsets > 2) return fail(ISSM_E_UNSUPPORTED, "dwconv: nsets = %d (1 or 2)", a->nsets);
  if (a->chain && a->nsets != 2) return fail(ISSM_E_SHAPE, "dwconv: chain needs nsets = 2, got %d", a->nsets);
  if (a->dtype != ISSM_F32 && a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "dwconv: dtype %d", a->dtype);
  if (!a->u || !a->w || (!a->pre && !heads_only)) return fail(ISSM_E_NULL, "dwconv: u/w/pre is NULL");
  if (a->u_token_stride < a->channels || a->u_batch_stride < 0)
    return fail(ISSM_E_STRIDE, "dwconv: u strides (%lld, %lld)", (long long)a->u_batch_stride, (long long)a->u_token_stride);
  if (!bwd && (!a->bias || !a->y)) return fail(ISSM_E_NULL, "dwconv: bias/y is NULL");
  if (bwd && (!a->partial || (!part && (!a->dw || !a->dbias)))) return fail(ISSM_E_NULL, "dwconv bwd: partial/dw/dbias is NULL");
  p->B = a->batch; p->L = a->seqlen; p->C = a->channels; p->nsets = a->nsets; p->dtype = a->dtype;
  p->chain = a->chain ? 1 : 0;
  p->u = a->u; p->u_bs = a->u_batch_stride; p->u_ls = a->u_token_stride;
  if (a->split < 0 || a->split >= a->channels) return fail(ISSM_E_SHAPE, "dwconv: split %d outside [0, channels)", a->split);
  if (a->split > 0 && !bwd && !a->y_tail && !heads_only) return fail(ISSM_E_NULL, "dwconv: y_tail is NULL");
  p->split = a->split; p->y_tail = a->y_tail;
  p->dy_tail[0] = a->dy_tail[0]; p->dy_tail[1] = a->nsets > 1 ? a->dy_tail[1] : nullptr;
  p->w = a->w; p->bias = a->bias; p->y = a->y; p->pre = a->pre;
  p->dy[0] = a->dy[0]; p->dy[1] = a->nsets > 1 ? a->dy[1] : nullptr;
  if ((a->du_batch_stride || a->du_token_stride) && (a->du_token_stride < a->channels || a->du_batch_stride < 0))
    return fail(ISSM_E_STRIDE, "dwconv: du strides (%lld, %lld)", (long long)a->du_batch_stride, (long long)a->du_token_stride);
  p->du = a->du; p->partial = a->partial; p->nrows = 0;
  p->du_ls = a->du_token_stride ? a->du_token_stride : a->channels;
  p->du_bs = a->du_token_stride ? a->du_batch_stride : (long)a->seqlen * a->channels;
  p->dw = a->dw; p->dbias = a->dbias;
  return ISSM_OK;
}

int issm_dwconv_partial_rows(int32_t batch, int32_t seqlen) {
  return (batch > 0 && seqlen > 0) ? dwconv_partial_rows(batch, seqlen, false) : 0;   // (a chained pair's are no more)
}

int issm_dwconv_part_rows(int32_t batch, int32_t seqlen) {
  return (batch > 0 && seqlen > 0) ? dwconv_partial_rows(batch, seqlen, true) : 0;
}

int issm_dwconv_silu_fwd(const issm_dwconv_args* a) {
  DwConvP p;
  int rc = dwconv_params(a, &p, false);
  if (rc) return rc;
  if (p.B == 0 || p.L == 0) return ISSM_OK;
  return launched(launch_dwconv_fwd(p, (hipStream_t)a->stream), "dwconv_silu_fwd");
}

int issm_conv_param_gen_fwd(const issm_dwconv_args* a, const issm_pgen_args* b) {
  DwConvP c;
  PGenP p;
  int rc = dwconv_params(a, &c, false, true);
  if (rc || (rc = pgen_params(b, &p, false, true, true))) return rc;
  if (c.dtype != ISSM_BF16 || p.dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "conv_param_gen: dtypes %d, %d (bf16 only)", c.dtype, p.dtype);
  if (!c.chain || p.bias || !p.has_back || c.split < 1 || c.C - c.split != 2 * p.G || p.tokens != (long)c.B * c.L)
    return fail(ISSM_E_SHAPE, "conv_param_gen: the two do not belong together (chain %d, split %d of %d, G %d, %lld and %d x %d tokens)",
                c.chain, c.split, c.C, p.G, (long long)p.tokens, c.B, c.L);
  if (p.tokens > 0x7fffffff) return fail(ISSM_E_SHAPE, "conv_param_gen: too large");
  if (p.tokens == 0) return ISSM_OK;
  if (p.K == 0) return fail(ISSM_E_SHAPE, "conv_param_gen: K = 0");
  p.dt_raw = nullptr;
  return launched(launch_conv_pgen(c, p, (hipStream_t)a->stream), "conv_param_gen_fwd");
}

int issm_dwconv_silu_bwd(const issm_dwconv_args* a) {
  DwConvP p;
  int rc = dwconv_params(a, &p, true);
  if (rc) return rc;
  return launched(launch_dwconv_bwd(p, (hipStream_t)a->stream), "dwconv_silu_bwd");
}

int issm_dwconv_silu_bwd_part(const issm_dwconv_args* a) {
  DwConvP p;
  int rc = dwconv_params(a, &p, true, false, true);
  if (rc) return rc;
  if (!p.chain) return fail(ISSM_E_UNSUPPORTED, "dwconv_bwd_part: a chained pair only");
  if (p.B == 0 || p.L == 0) return ISSM_OK;
  p.dw = p.dbias = nullptr;
  return launched(launch_dwconv_bwd(p, (hipStream_t)a->stream), "dwconv_silu_bwd_part");
}

static int box_dist_params(const issm_box_dist_args* a, BoxDistP* p, bool bwd) {
  if (!a) return fail(ISSM_E_NULL, "box_dist: args is NULL");
  if (a->batch < 0 || a->seqlen < 0 || a->nquery < 0 || a->D < 1 || a->H < 1 || a->W < 1)
    return fail(ISSM_E_SHAPE, "box_dist: bad shape");
  if ((int64_t)a->D * a->H * a->W > 1024)
    return fail(ISSM_E_UNSUPPORTED, "box_dist: table of %d x %d x %d nodes (at most 1024 fit)", a->D, a->H, a->W);
  if (a->dtype != ISSM_F32 && a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "box_dist: dtype %d", a->dtype);
  if (!a->key || (!a->corners && !a->boxes)) return fail(ISSM_E_NULL, "box_dist: key or corners/boxes is NULL");
  if (!bwd) {
    if (a->dist && !a->table) return fail(ISSM_E_NULL, "box_dist: table is NULL");
    if (a->weights && !a->boxes && (!a->qcenter || !a->radius)) return fail(ISSM_E_NULL, "box_dist: qcenter/radius is NULL");
    if (a->qcenter && !a->radius) return fail(ISSM_E_NULL, "box_dist: radius is NULL");
  } else if (!a->ddist || !a->partial || !a->dtable) {
    return fail(ISSM_E_NULL, "box_dist bwd: ddist/partial/dtable is NULL");
  }
  p->B = a->batch; p->L = a->seqlen; p->K = a->nquery; p->D = a->D; p->H = a->H; p->W = a->W; p->dtype = a->dtype;
  p->nwg = box_dist_workgroups(a->batch, a->seqlen, a->nquery);
  p->nwg_bwd = box_dist_bwd_workgroups(a->batch, a->seqlen, a->nquery);
  if (bwd && (int64_t)a->batch * a->seqlen * a->nquery > ((int64_t)1 << 26))
    return fail(ISSM_E_UNSUPPORTED, "box_dist bwd: more than 2^26 (point, box) pairs");
  p->key = a->key; p->corners = a->corners; p->boxes = a->corners ? nullptr : a->boxes; p->min_radius = a->min_radius;
  p->angle = a->angle; p->table = a->table;
  p->log_scale = a->log_scale; p->max_value = a->max_value; p->dist = a->dist;
  p->qcenter = a->qcenter; p->radius = a->radius; p->weight_dist = a->weight_dist; p->weights = a->weights;
  p->ddist = a->ddist; p->partial = a->partial; p->dtable = a->dtable;
  return ISSM_OK;
}

int64_t issm_box_dist_bwd_scratch_bytes(int32_t batch, int32_t seqlen, int32_t nquery, int32_t D, int32_t H, int32_t W) {
  if (batch <= 0 || seqlen <= 0 || nquery <= 0 || D <= 0 || H <= 0 || W <= 0) return 16;
  return box_dist_bwd_scratch_bytes(batch, seqlen, nquery, D, H, W);
}

static int box_table_params(const issm_box_table_args* a, BoxTableP& p) {
  if (!a) return fail(ISSM_E_NULL, "box_table: args is NULL");
  if (a->nodes < 1 || a->hidden < 1 || a->nodes > (1 << 26)) return fail(ISSM_E_SHAPE, "box_table: %d nodes, %d hidden", a->nodes, a->hidden);
  if (a->hidden > 256) return fail(ISSM_E_UNSUPPORTED, "box_table: %d hidden values (at most 256)", a->hidden);
  for (int t : {a->dtype, a->coords_dtype})
    if (t != ISSM_F32 && t != ISSM_BF16) return fail(ISSM_E_DTYPE, "box_table: dtype %d", t);
  if (!a->coords || !a->w1 || !a->b1 || !a->w2) return fail(ISSM_E_NULL, "box_table: coords/w1/b1/w2 is NULL");
  p = BoxTableP{a->nodes, a->hidden, a->dtype, a->coords_dtype, a->coords, a->w1, a->b1, a->w2, a->table};
  return ISSM_OK;
}

int issm_box_table_bwd(const issm_box_table_args* a, const float* dtable, void* dw1, void* db1, void* dw2) {
  BoxTableP p;
  if (const int rc = box_table_params(a, p)) return rc;
  if (!dtable || !dw1 || !db1 || !dw2) return fail(ISSM_E_NULL, "box_table_bwd: dtable/dw1/db1/dw2 is NULL");
  return launched(launch_box_table_bwd(p, dtable, dw1, db1, dw2, (hipStream_t)a->stream), "box_table_bwd");
}

int issm_box_table(const issm_box_table_args* a) {
  BoxTableP p;
  if (const int rc = box_table_params(a, p)) return rc;
  if (!p.table) return fail(ISSM_E_NULL, "box_table: table is NULL");
  return launched(launch_box_table(p, (hipStream_t)a->stream), "box_table");
}

static int box_dist_fwd(const issm_box_dist_args* a, bool only) {
  BoxDistP p;
  int rc = box_dist_params(a, &p, false);
  if (rc) return rc;
  if (p.nwg == 0 || (!p.dist && !p.weights)) return ISSM_OK;
  return launched(launch_box_dist_fwd(p, only, (hipStream_t)a->stream), "box_dist_fwd");
}
int issm_box_dist_fwd(const issm_box_dist_args* a) { return box_dist_fwd(a, false); }
int issm_box_dist_fwd_only(const issm_box_dist_args* a) { return box_dist_fwd(a, true); }

int issm_box_dist_bwd(const issm_box_dist_args* a) {
  BoxDistP p;
  int rc = box_dist_params(a, &p, true);
  if (rc) return rc;
  if (p.nwg_bwd == 0) return ISSM_OK;
  return launched(launch_box_dist_bwd(p, (hipStream_t)a->stream), "box_dist_bwd");
}

static int layer_params(const issm_layer_params_args* a, LayerParamsP& p) {
  static_assert(LAYER_ARRAYS == ISSM_LAYER_ARRAYS, "one count");
  if (!a) return fail(ISSM_E_NULL, "layer_params: args is NULL");
  if (a->a_log < 0 || a->a_log >= LAYER_ARRAYS || a->K < 0) return fail(ISSM_E_SHAPE, "layer_params: a_log %d, K %d", a->a_log, a->K);
  int64_t total = 0;
  for (int i = 0; i < LAYER_ARRAYS; ++i) {
    if (a->n[i] < 0) return fail(ISSM_E_SHAPE, "layer_params: n[%d] = %d", i, a->n[i]);
    if (a->dtype[i] != ISSM_F32 && a->dtype[i] != ISSM_BF16) return fail(ISSM_E_DTYPE, "layer_params: dtype[%d] = %d", i, a->dtype[i]);
    if (a->n[i] && !a->src[i]) return fail(ISSM_E_NULL, "layer_params: src[%d] is NULL", i);
    p.src[i] = a->src[i]; p.n[i] = a->n[i]; p.bf16[i] = a->dtype[i] == ISSM_BF16;
    total += a->n[i];
  }
  p.a_log = a->a_log; p.H = a->n[a->a_log]; p.K = a->K; p.out = a->out; p.A = a->A;
  if (total + (int64_t)p.H * p.K > ((int64_t)1 << 30)) return fail(ISSM_E_SHAPE, "layer_params: too large");
  p.total = (int)total;
  if (total && (!a->out || !a->A)) return fail(ISSM_E_NULL, "layer_params: out/A is NULL");
  return ISSM_OK;
}

int issm_layer_params(const issm_layer_params_args* a) {
  LayerParamsP p;
  const int rc = layer_params(a, p);
  if (rc || p.total == 0) return rc;
  return launched(launch_layer_params(p, (hipStream_t)a->stream), "layer_params");
}

static int linear_params(const issm_linear_args* a, LinearP& p, int& n) {
  if (!a) return fail(ISSM_E_NULL, "linear: args is NULL");
  if (a->njobs < 0 || a->njobs > ISSM_LINEAR_JOBS) return fail(ISSM_E_SHAPE, "linear: %d products (0..%d)", a->njobs, ISSM_LINEAR_JOBS);
  if (a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "linear: dtype %d (bf16 only)", a->dtype);
  n = 0;
  for (int i = 0; i < a->njobs; ++i) {
    const issm_linear_job& j = a->job[i];
    if (j.tokens < 0 || j.in < 0 || j.out < 0 || j.tokens > 0x7fffffff - 64 || j.out > 0x7fffffff - 64)
      return fail(ISSM_E_SHAPE, "linear: (%lld, %d) -> %d", (long long)j.tokens, j.in, j.out);
    if (j.in == 0 || j.in % 32) return fail(ISSM_E_UNSUPPORTED, "linear: %d features (a multiple of 32)", j.in);
    if (j.tokens == 0 || j.out == 0) continue;
    if (!j.x || !j.w || !j.y) return fail(ISSM_E_NULL, "linear: x/w/y is NULL");
    if (((uintptr_t)j.x | (uintptr_t)j.w) & 15) return fail(ISSM_E_STRIDE, "linear: x and w must be aligned to 16 bytes");
    if ((uintptr_t)j.y & 1) return fail(ISSM_E_STRIDE, "linear: y must be aligned to its elements");
    if (j.turn < 0 || (j.turn && j.tokens % j.turn)) return fail(ISSM_E_SHAPE, "linear: %lld tokens, turned by %d", (long long)j.tokens, j.turn);
    p.job[n++] = LinearJob{(const uint16_t*)j.x, (const uint16_t*)j.w, (uint16_t*)j.y, (int)j.tokens, j.out, j.in / 32, 0, j.turn};
  }
  return ISSM_OK;
}

// Which products of a launch go through LDS in tiles (linear_tile.hip), the others straight from memory into the matrix operands (linear.hip): the
// same sums in the same order.  Tiles from 64 tokens and 96 outputs on, each product for itself (linear.hip and tiles in us: 1024 x 96 -> 202 3.4 and 2.9,
// 192 -> 394 4.8 and 3.8, 320 -> 650 12.9 and 5.1, 4096 x 288 -> 586 11.4 and 6.0; beside 32 x 288 -> 288, 8192 x 288 -> 586 20.7 and 10.2, beside 63 x 192 -> 192,
// 512 x 192 -> 192 4.7 and 4.7), but for odd multiples of 288 features, nine fragments from rows that lie across the memory channels, which linear.hip
// has sooner as long as a launch's workgroups there have a CU each: 288 -> 288 of 1024, 1536 and 2048 tokens (144, 216 and 288 workgroups) 3.8 and 4.4,
// 3.8 and 4.4, 5.4 and 4.5; 768 and 1024 x 288 -> 586 (228 and 304) 3.9 and 4.5, 5.6 and 4.5; 1024 x 288 -> 288 beside 512 and 1024 tokens (216 and 288) 3.9 and
// 4.4, 5.5 and 4.4; 864 -> 288 of 1536 and 2048 tokens 7.7 and 8.4, 13.1 and 8.5 (of 576 features tiles are ahead from 64 tokens on, 8.0 and 6.3).
static void linear_forms(const LinearP& p, int n, bool (&tiles)[2]) {
  int64_t workgroups = 0;
  bool nines = true;
  for (int i = 0; i < n; ++i) {
    const LinearJob& j = p.job[i];
    tiles[i] = !j.turn && linear_tile_takes(j.tokens, 32 * j.steps, j.out, false);
    workgroups += ((int64_t)j.tokens + 63) / 64 * (((int64_t)j.out + 31) / 32);
    nines = nines && j.steps % 18 == 9;
  }
  if (nines && workgroups <= NCU) tiles[0] = tiles[1] = false;
}
static LinearTileJob linear_tile_job(const LinearJob& j) { return LinearTileJob{j.x, j.w, j.y, j.tokens, 32 * j.steps, j.out, 0}; }

int issm_linear_fwd(const issm_linear_args* a) {
  LinearP p{};
  int n;
  const int rc = linear_params(a, p, n);
  if (rc || n == 0) return rc;
  bool tiles[2] = {false, false};
  linear_forms(p, n, tiles);
  LinearTileP q{};
  if (n == 2 && tiles[0] != tiles[1]) {   // the tiles first
    if (tiles[1]) std::swap(p.job[0], p.job[1]);
    q.job[0] = linear_tile_job(p.job[0]);
    return launched(launch_layer_in_tile(q, p, LayerParamsP{}, (hipStream_t)a->stream), "linear_fwd");
  }
  if (tiles[0]) {
    for (int i = 0; i < n; ++i) q.job[i] = linear_tile_job(p.job[i]);
    return launched(launch_linear_tile(q, n, false, (hipStream_t)a->stream), "linear_fwd");
  }
  return launched(launch_linear(p, n, nullptr, (hipStream_t)a->stream), "linear_fwd");
}

int issm_linear_dx(const issm_linear_args* a) {
  if (!a) return fail(ISSM_E_NULL, "linear_dx: args is NULL");
  if (a->njobs < 0 || a->njobs > ISSM_LINEAR_JOBS) return fail(ISSM_E_SHAPE, "linear_dx: %d products (0..%d)", a->njobs, ISSM_LINEAR_JOBS);
  if (a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "linear_dx: dtype %d (bf16 only)", a->dtype);
  LinearTileP p{};
  for (int i = 0; i < a->njobs; ++i) {
    const issm_linear_job& j = a->job[i];
    if (j.tokens < 0 || j.in < 0 || j.out < 0 || j.turn || j.tokens > 0x7fffffff - 64)
      return fail(ISSM_E_SHAPE, "linear_dx: (%lld, %d) -> %d, turned by %d", (long long)j.tokens, j.in, j.out, j.turn);
    if (!linear_tile_takes(j.tokens, j.in, j.out, true))
      return fail(ISSM_E_UNSUPPORTED, "linear_dx: (%lld, %d) -> %d (from 64 tokens and 96 results on, even sizes)", (long long)j.tokens, j.in, j.out);
    if (!j.x || !j.w || !j.y) return fail(ISSM_E_NULL, "linear_dx: x/w/y is NULL");
    if (((uintptr_t)j.x | (uintptr_t)j.w) & 3) return fail(ISSM_E_STRIDE, "linear_dx: x and w must be aligned to 4 bytes");
    if ((uintptr_t)j.y & 1) return fail(ISSM_E_STRIDE, "linear_dx: y must be aligned to its elements");
    p.job[i] = LinearTileJob{(const uint16_t*)j.x, (const uint16_t*)j.w, (uint16_t*)j.y, (int)j.tokens, j.in, j.out, 0};
  }
  if (a->njobs == 0) return ISSM_OK;
  return launched(launch_linear_tile(p, a->njobs, true, (hipStream_t)a->stream), "linear_dx");
}

int issm_layer_in(const issm_linear_args* a, const issm_layer_params_args* b) {
  LinearP p{};
  LayerParamsP q;
  int n, rc = linear_params(a, p, n);
  if (rc || (rc = layer_params(b, q))) return rc;
  if (n == 0 || q.total == 0) {   // (nothing to join)
    if (n && (rc = issm_linear_fwd(a))) return rc;
    return q.total ? issm_layer_params(b) : ISSM_OK;
  }
  bool tiles[2];
  linear_forms(p, n, tiles);
  if (tiles[0]) {
    LinearTileP t{};
    t.job[0] = linear_tile_job(p.job[0]);
    return launched(launch_layer_in_tile(t, p, q, (hipStream_t)a->stream), "layer_in");
  }
  return launched(launch_linear(p, n, &q, (hipStream_t)a->stream), "layer_in");
}

static bool linear_dw_sizes(int64_t tokens, int32_t in, int32_t out) {
  return tokens >= 0 && tokens <= 0x7fffffff / 2 && in >= 6 && out >= 4 && (int64_t)in * out < ((int64_t)1 << 31);
}

size_t issm_linear_dw_scratch_bytes(int64_t tokens, int32_t in, int32_t out) {
  return linear_dw_sizes(tokens, in, out) ? (size_t)linear_dw_splits(tokens, in, out) * in * out * sizeof(float) : 0;
}

static int linear_dw_params(const issm_linear_dw_args* a, LinearDwP& p) {
  if (!a) return fail(ISSM_E_NULL, "linear_dw: args is NULL");
  if (a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "linear_dw: dtype %d (bf16 only)", a->dtype);
  if (!linear_dw_sizes(a->tokens, a->in, a->out)) return fail(ISSM_E_SHAPE, "linear_dw: %lld tokens, (%d, %d)", (long long)a->tokens, a->out, a->in);
  if (a->tokens == 0) return fail(ISSM_E_SHAPE, "linear_dw: no tokens");
  if (!a->dy || !a->x || !a->dw || !a->scratch) return fail(ISSM_E_NULL, "linear_dw: dy/x/dw/scratch is NULL");
  if (a->scratch_bytes < issm_linear_dw_scratch_bytes(a->tokens, a->in, a->out)) return fail(ISSM_E_WORKSPACE, "linear_dw: scratch too small");
  if ((uintptr_t)a->scratch & 15) return fail(ISSM_E_STRIDE, "linear_dw: scratch must be aligned to 16 bytes");
  if (((uintptr_t)a->dy | (uintptr_t)a->x | (uintptr_t)a->dw) & 1) return fail(ISSM_E_STRIDE, "linear_dw: operands must be aligned to their elements");
  p.dy = (const uint16_t*)a->dy; p.x = (const uint16_t*)a->x; p.dw = (uint16_t*)a->dw; p.partial = (float*)a->scratch;
  p.tokens = (int)a->tokens; p.in = a->in; p.out = a->out;
  p.splits = linear_dw_splits(a->tokens, a->in, a->out);
  return ISSM_OK;
}

int issm_linear_dw(const issm_linear_dw_args* a) {
  LinearDwJobs j{};
  if (const int rc = linear_dw_params(a, j.job[0])) return rc;
  return launched(launch_linear_dw(j, 1, (hipStream_t)a->stream), "linear_dw");
}

int issm_linear_dw_pair(const issm_linear_dw_args* a, const issm_linear_dw_args* b) {
  LinearDwJobs j{};
  int rc = linear_dw_params(a, j.job[0]);
  if (rc || (rc = linear_dw_params(b, j.job[1]))) return rc;
  return launched(launch_linear_dw(j, 2, (hipStream_t)a->stream), "linear_dw_pair");
}

static int layer_out_params(const issm_layer_out_args* a, LayerOutP& p, bool norms_out) {
  if (!a) return fail(ISSM_E_NULL, "layer_out: args is NULL");
  if (a->batch < 0 || a->seqlen < 0 || a->queries < 0 || a->d_inner < 1) return fail(ISSM_E_SHAPE, "layer_out: bad shape");
  if (a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "layer_out: dtype %d (bf16 only)", a->dtype);
  if (a->d_inner % 4 || a->d_inner > 1024)
    return fail(ISSM_E_UNSUPPORTED, "layer_out: %d features (a multiple of 4, at most 1024)", a->d_inner);
  p.rows = (long)a->batch * a->seqlen;
  p.B = a->queries ? a->batch : 0;
  p.K = a->queries ? a->queries : 1;
  if (p.rows && (!a->y[0] || !a->y[1] || !a->z || !a->key_weight || (norms_out && !a->key)))
    return fail(ISSM_E_NULL, "layer_out: y/z/key_weight/key is NULL");
  if (p.rows && a->z_row_stride < a->d_inner) return fail(ISSM_E_STRIDE, "layer_out: z_row_stride %lld", (long long)a->z_row_stride);
  if (p.B && (!a->last[0] || !a->last[1] || (norms_out && !a->query))) return fail(ISSM_E_NULL, "layer_out: last/query is NULL");
  p.y0 = (const uint16_t*)a->y[0]; p.y1 = (const uint16_t*)a->y[1]; p.z = (const uint16_t*)a->z; p.zs = a->z_row_stride;
  p.kw = (const uint16_t*)a->key_weight; p.qw = (const uint16_t*)a->query_weight; p.qb = (const uint16_t*)a->query_bias;
  p.key = (uint16_t*)a->key; p.query = (uint16_t*)a->query;
  p.last0 = a->last[0]; p.last1 = a->last[1];
  p.di = a->d_inner; p.keps = a->key_eps; p.qeps = a->query_eps;
  return ISSM_OK;
}

int issm_layer_out(const issm_layer_out_args* a) {
  LayerOutP p{};
  const int rc = layer_out_params(a, p, true);
  if (rc || (p.rows == 0 && p.B == 0)) return rc;
  return launched(launch_layer_out(p, (hipStream_t)a->stream), "layer_out");
}

int issm_layer_end(const issm_layer_out_args* a, const issm_linear_args* b) {
  LayerOutP p{};
  LinearP q{};
  const int rc = layer_out_params(a, p, false);
  if (rc) return rc;
  if (!b) return fail(ISSM_E_NULL, "layer_end: products is NULL");
  if (b->njobs != 2) return fail(ISSM_E_SHAPE, "layer_end: %d products (2)", b->njobs);
  if (b->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "layer_end: dtype %d (bf16 only)", b->dtype);
  if (p.di % 32) return fail(ISSM_E_UNSUPPORTED, "layer_end: %d features (a multiple of 32)", p.di);
  for (int i = 0; i < 2; ++i) {
    const issm_linear_job& j = b->job[i];
    const long rows = i ? (long)p.B * p.K : p.rows;
    if (j.tokens != rows || j.in != p.di || j.out < 0 || j.out > 0x7fffffff - 128 || j.turn || rows > 0x7fffffff - 64)
      return fail(ISSM_E_SHAPE, "layer_end: product %d of (%lld, %d) -> %d, turned by %d", i, (long long)j.tokens, j.in, j.out, j.turn);
    const int out = rows ? j.out : 0;
    if (out && (!j.w || !j.y)) return fail(ISSM_E_NULL, "layer_end: w/y is NULL");
    if (out && (((uintptr_t)j.w & 15) || ((uintptr_t)j.y & 1))) return fail(ISSM_E_STRIDE, "layer_end: w must be aligned to 16 bytes, y to its elements");
    q.job[i] = LinearJob{nullptr, (const uint16_t*)j.w, (uint16_t*)j.y, (int)rows, out, p.di / 32, 0, 0};
  }
  return launched(launch_layer_end(p, q, (hipStream_t)a->stream), "layer_end");
}

static int transpose_params(const issm_transpose_args* a, TrP& p) {
  if (!a) return fail(ISSM_E_NULL, "transpose: args is NULL");
  if (a->batch < 0 || a->rows < 0 || a->cols < 0) return fail(ISSM_E_SHAPE, "transpose: bad shape");
  if ((a->in_dtype != ISSM_F32 && a->in_dtype != ISSM_BF16) || (a->out_dtype != ISSM_F32 && a->out_dtype != ISSM_BF16))
    return fail(ISSM_E_DTYPE, "transpose: dtypes %d -> %d", a->in_dtype, a->out_dtype);
  p.B = 0;
  if (a->batch == 0 || a->rows == 0 || a->cols == 0) return ISSM_OK;
  if (!a->in0 || !a->out) return fail(ISSM_E_NULL, "transpose: in0/out is NULL");
  if (a->batch > 65535 || (a->rows + 63) / 64 > 65535) return fail(ISSM_E_SHAPE, "transpose: batch / rows too large for one launch");
  p.B = a->batch; p.R = a->rows; p.C = a->cols; p.in_dt = a->in_dtype; p.out_dt = a->out_dtype;
  p.in0 = a->in0; p.in1 = a->in1; p.out = a->out; p.alpha = a->alpha;
  return ISSM_OK;
}

int issm_transpose_states(const issm_transpose_args* a) {
  TrP p;
  const int rc = transpose_params(a, p);
  if (rc || p.B == 0) return rc;
  return launched(launch_transpose_states(p, (hipStream_t)a->stream), "transpose_states");
}

int issm_layer_begin(const issm_layer_params_args* a, const issm_transpose_args* b) {
  LayerParamsP p;
  TrP t{};
  int rc = layer_params(a, p);
  if (rc || (rc = transpose_params(b, t))) return rc;
  if (b->in_dtype != b->out_dtype) return fail(ISSM_E_UNSUPPORTED, "layer_begin: states of one type");
  if (p.total == 0 && t.B == 0) return ISSM_OK;
  return launched(launch_layer_begin(p, t, (hipStream_t)a->stream), "layer_begin");
}

int issm_layer_behind(const issm_norm_args* a, const void* x2, void* sum, const issm_transpose_args* b) {
  NormP p;
  TrP t{};
  int rc = norm_params(a, &p, false);
  if (rc || (rc = transpose_params(b, t))) return rc;
  if (!x2 || !sum) return fail(ISSM_E_NULL, "layer_behind: x2/sum is NULL");
  if (b->in_dtype != ISSM_F32 || !layer_behind_takes(p) || p.xs != p.ncols)
    return fail(ISSM_E_UNSUPPORTED, "layer_behind: one group of up to 1024 columns, a multiple of 4, in contiguous rows, no bias, fp32 states");
  norm_scratch_warm((hipStream_t)a->stream);
  return launched(launch_layer_behind(p, x2, sum, t, (hipStream_t)a->stream), "layer_behind");
}

int issm_layer_grads(const issm_layer_grads_args* a, const issm_transpose_args* b) {
  if (!a) return fail(ISSM_E_NULL, "layer_grads: args is NULL");
  if (a->conv_rows < 0 || a->gen_rows < 0 || a->norm_rows < 0 || a->C < 1 || a->H < 1 || a->G < 1 || a->d_inner < 1 || a->K < 0 || a->nD < 0)
    return fail(ISSM_E_SHAPE, "layer_grads: bad shape");
  if (a->dtype != ISSM_F32 && a->dtype != ISSM_BF16) return fail(ISSM_E_DTYPE, "layer_grads: dtype %d", a->dtype);
  if (((int64_t)a->C + a->H + a->G) * 64 + (int64_t)a->H * a->K + a->d_inner + a->nD > ((int64_t)1 << 30)) return fail(ISSM_E_SHAPE, "layer_grads: too large");
  if ((a->conv_rows && !a->conv) || (a->gen_rows && !a->gen) || (a->norm_rows && !a->norm) || (a->K && (!a->dA || !a->A)) || (a->nD && !a->dD) || !a->out)
    return fail(ISSM_E_NULL, "layer_grads: a part or out is NULL");
  TrP t{};
  if (b) {
    const int rc = transpose_params(b, t);
    if (rc) return rc;
    if (b->in_dtype != ISSM_F32 || b->in1) return fail(ISSM_E_UNSUPPORTED, "layer_grads: states are one fp32 tensor");
  }
  const long R0 = a->H + 2 * a->G;
  LayerGradsP p{};
  p.conv = a->conv; p.gen = a->gen; p.gen_bias = a->gen ? a->gen + a->gen_rows * R0 * 16 : nullptr; p.norm = a->norm;
  p.conv_rows = a->conv_rows; p.gen_rows = a->gen_rows; p.norm_rows = a->norm_rows;
  p.C = a->C; p.H = a->H; p.R0 = (int)R0; p.di = a->d_inner; p.K = a->K; p.nD = a->nD;
  p.dA = a->dA; p.A = a->A; p.dD = a->dD; p.out = a->out; p.bf16 = a->dtype == ISSM_BF16;
  return launched(launch_layer_grads(p, t, (hipStream_t)a->stream), "layer_grads");
}

int issm_hilbert_codes(const issm_hilbert_args* a) {
  if (!a) return fail(ISSM_E_NULL, "hilbert: args is NULL");
  if (a->batch < 0 || a->npoint < 0) return fail(ISSM_E_SHAPE, "hilbert: bad shape");
  if (a->bits < 1 || a->bits > 20) return fail(ISSM_E_UNSUPPORTED, "hilbert: bits = %d (1..20)", a->bits);
  if (!(a->cell > 0.0f)) return fail(ISSM_E_SHAPE, "hilbert: cell must be positive");
  int seen = 0;
  for (int i = 0; i < 3; ++i) {
    if (a->order[i] < 0 || a->order[i] > 2) return fail(ISSM_E_SHAPE, "hilbert: order[%d] = %d", i, a->order[i]);
    seen |= 1 << a->order[i];
  }
  if (seen != 7) return fail(ISSM_E_SHAPE, "hilbert: order is not a permutation of 0, 1, 2");
  if ((int64_t)a->batch * a->npoint == 0) return ISSM_OK;
  if (!a->points || !a->mins || !a->codes) return fail(ISSM_E_NULL, "hilbert: points/mins/codes is NULL");
  HilbertP p;
  p.B = a->batch; p.N = a->npoint; p.bits = a->bits; p.cell = a->cell;
  for (int i = 0; i < 3; ++i) p.perm[i] = a->order[i];
  p.points = a->points; p.mins = a->mins; p.codes = (long*)a->codes;
  return launched(launch_hilbert_codes(p, (hipStream_t)a->stream), "hilbert_codes");
}

int issm_hilbert_order(const issm_hilbert_order_args* a) {
  if (!a) return fail(ISSM_E_NULL, "hilbert_order: args is NULL");
  if (a->batch < 0 || a->npoint < 0) return fail(ISSM_E_SHAPE, "hilbert_order: bad shape");
  if (a->norder < 1 || a->norder > 6) return fail(ISSM_E_SHAPE, "hilbert_order: norder = %d (1..6)", a->norder);
  if (a->bits < 1 || a->bits > 17) return fail(ISSM_E_UNSUPPORTED, "hilbert_order: bits = %d (1..17)", a->bits);
  if (a->npoint > ISSM_HILBERT_ORDER_MAX_POINTS)
    return fail(ISSM_E_UNSUPPORTED, "hilbert_order: %d points (at most %d per sample; use issm_hilbert_codes and a sort)",
                a->npoint, ISSM_HILBERT_ORDER_MAX_POINTS);
  if (!(a->cell > 0.0f)) return fail(ISSM_E_SHAPE, "hilbert_order: cell must be positive");
  for (int o = 0; o < a->norder; ++o) {
    int seen = 0;
    for (int i = 0; i < 3; ++i) {
      if (a->order[o][i] < 0 || a->order[o][i] > 2) return fail(ISSM_E_SHAPE, "hilbert_order: order[%d][%d] = %d", o, i, a->order[o][i]);
      seen |= 1 << a->order[o][i];
    }
    if (seen != 7) return fail(ISSM_E_SHAPE, "hilbert_order: order %d is not a permutation of 0, 1, 2", o);
  }
  if ((int64_t)a->batch * a->npoint == 0) return ISSM_OK;
  if (!a->points || !a->index) return fail(ISSM_E_NULL, "hilbert_order: points/index is NULL");
  if ((int64_t)a->batch * a->norder > 0x7fffffff) return fail(ISSM_E_SHAPE, "hilbert_order: too many samples");
  HilbertOrderP p;
  p.B = a->batch; p.N = a->npoint; p.bits = a->bits; p.norder = a->norder; p.cell = a->cell;
  p.NP = 2;
  while (p.NP < p.N) p.NP <<= 1;
  for (int o = 0; o < a->norder; ++o)
    for (int i = 0; i < 3; ++i) p.perm[o][i] = a->order[o][i];
  p.points = a->points; p.index = (long*)a->index; p.inverse = (long*)a->inverse;
  return launched(launch_hilbert_order(p, (hipStream_t)a->stream), "hilbert_order");
}

// shared checks of the point-set operators: non-negative sizes, work present, pointers given
#define PN2_SIZES(what, ...)                                                              \
  do {                                                                                    \
    const long long dims_[] = {__VA_ARGS__};                                              \
    for (long long d_ : dims_)                                                            \
      if (d_ < 0) return fail(ISSM_E_SHAPE, what ": negative size");                      \
  } while (0)
#define PN2_PTRS(what, ...)                                                               \
  do {                                                                                    \
    const void* ptrs_[] = {__VA_ARGS__};                                                  \
    for (const void* q_ : ptrs_)                                                          \
      if (!q_) return fail(ISSM_E_NULL, what ": NULL pointer");                           \
  } while (0)

int issm_pn2_furthest_point_sampling(int32_t b, int32_t n, int32_t npoint, const float* xyz, float* temp, int32_t* idxs,
                                     void* stream) {
  PN2_SIZES("furthest_point_sampling", b, n, npoint);
  if (b == 0 || npoint == 0) return ISSM_OK;
  if (n == 0) return fail(ISSM_E_SHAPE, "furthest_point_sampling: no points to draw from");
  if (b > 65535) return fail(ISSM_E_UNSUPPORTED, "furthest_point_sampling: batch %d > 65535", b);
  PN2_PTRS("furthest_point_sampling", xyz, idxs);
  if (n > 24576 && !temp) return fail(ISSM_E_NULL, "furthest_point_sampling: temp is NULL (needed above 24576 points)");
  return launched(launch_fps(b, n, npoint, xyz, temp, idxs, (hipStream_t)stream), "furthest_point_sampling");
}

int issm_pn2_ball_query(int32_t b, int32_t n, int32_t m, float radius, int32_t nsample, const float* new_xyz,
                        const float* xyz, int32_t* idx, void* stream) {
  PN2_SIZES("ball_query", b, n, m, nsample);
  if (b == 0 || m == 0 || nsample == 0) return ISSM_OK;
  if (b > 65535) return fail(ISSM_E_UNSUPPORTED, "ball_query: batch %d > 65535", b);
  PN2_PTRS("ball_query", new_xyz, idx);
  if (n > 0 && !xyz) return fail(ISSM_E_NULL, "ball_query: xyz is NULL");
  return launched(launch_ball_query(b, n, m, radius, nsample, new_xyz, xyz, idx, (hipStream_t)stream), "ball_query");
}

int issm_pn2_group_points(int32_t b, int32_t c, int32_t n, int32_t npoints, int32_t nsample, const float* points,
                          const int32_t* idx, float* out, void* stream) {
  PN2_SIZES("group_points", b, c, n, npoints, nsample);
  if ((int64_t)b * c * npoints * nsample == 0) return ISSM_OK;
  if (n == 0) return fail(ISSM_E_SHAPE, "group_points: no points to index");
  if ((int64_t)npoints * nsample > 0x7fffffff) return fail(ISSM_E_SHAPE, "group_points: too many indices per sample");
  PN2_PTRS("group_points", points, idx, out);
  return launched(launch_group_points(b, c, n, npoints, nsample, nullptr, nullptr, 0.0f, points, idx, out, (hipStream_t)stream),
                  "group_points");
}

int issm_pn2_group_xyz_points(int32_t b, int32_t c, int32_t n, int32_t npoints, int32_t nsample, const float* xyz,
                              const float* new_xyz, float scale, const float* points, const int32_t* idx, float* out,
                              void* stream) {
  PN2_SIZES("group_xyz_points", b, c, n, npoints, nsample);
  if ((int64_t)b * npoints * nsample == 0) return ISSM_OK;
  if (n == 0) return fail(ISSM_E_SHAPE, "group_xyz_points: no points to index");
  if ((int64_t)npoints * nsample > 0x7fffffff) return fail(ISSM_E_SHAPE, "group_xyz_points: too many indices per sample");
  PN2_PTRS("group_xyz_points", xyz, new_xyz, idx, out);
  if (c > 0 && !points) return fail(ISSM_E_NULL, "group_xyz_points: points is NULL");
  return launched(launch_group_points(b, c, n, npoints, nsample, xyz, new_xyz, scale, points, idx, out, (hipStream_t)stream),
                  "group_xyz_points");
}

int issm_pn2_group_points_grad_rows(int32_t b, int32_t c, int32_t c0, int32_t cdim, int32_t n, int32_t npoints, int32_t nsample,
                                    const float* grad_out, const int32_t* idx, float* grad_points, void* stream) {
  PN2_SIZES("group_points_grad_rows", b, c, c0, cdim, n, npoints, nsample);
  if ((int64_t)b * c * npoints * nsample == 0) return ISSM_OK;
  if (n == 0 || (int64_t)c0 + c > cdim) return fail(ISSM_E_SHAPE, "group_points_grad_rows: no points, or channels beyond grad_out's");
  if (n > ISSM_PN2_ROW_POINTS || (int64_t)npoints * nsample > 0x7fffffff || (int64_t)b * c > 0x7fffffff / 1024)
    return fail(ISSM_E_UNSUPPORTED, "group_points_grad_rows: n = %d > %d, or too many indices or rows", n, ISSM_PN2_ROW_POINTS);
  PN2_PTRS("group_points_grad_rows", grad_out, idx, grad_points);
  return launched(launch_group_rows_grad(b, c, c0, cdim, n, npoints * nsample, grad_out, idx, grad_points, (hipStream_t)stream),
                  "group_points_grad_rows");
}

int issm_pn2_group_points_grad(int32_t b, int32_t c, int32_t n, int32_t npoints, int32_t nsample, const float* grad_out,
                               const int32_t* idx, float* grad_points, void* stream) {
  PN2_SIZES("group_points_grad", b, c, n, npoints, nsample);
  if ((int64_t)b * c * npoints * nsample == 0) return ISSM_OK;
  if (n == 0) return fail(ISSM_E_SHAPE, "group_points_grad: no points to index");
  if ((int64_t)npoints * nsample > 0x7fffffff) return fail(ISSM_E_SHAPE, "group_points_grad: too many indices per sample");
  PN2_PTRS("group_points_grad", grad_out, idx, grad_points);
  return launched(launch_group_points_grad(b, c, n, npoints * nsample, grad_out, idx, grad_points, (hipStream_t)stream),
                  "group_points_grad");
}

int issm_pn2_gather_points(int32_t b, int32_t c, int32_t n, int32_t npoints, const float* points, const int32_t* idx,
                           float* out, void* stream) {
  return issm_pn2_group_points(b, c, n, npoints, 1, points, idx, out, stream);
}

int issm_pn2_gather_points_grad(int32_t b, int32_t c, int32_t n, int32_t npoints, const float* grad_out,
                                const int32_t* idx, float* grad_points, void* stream) {
  return issm_pn2_group_points_grad(b, c, n, npoints, 1, grad_out, idx, grad_points, stream);
}

int issm_pn2_three_nn(int32_t b, int32_t n, int32_t m, const float* unknown, const float* known, float* dist2,
                      int32_t* idx, void* stream) {
  PN2_SIZES("three_nn", b, n, m);
  if (b == 0 || n == 0) return ISSM_OK;
  if (b > 65535) return fail(ISSM_E_UNSUPPORTED, "three_nn: batch %d > 65535", b);
  PN2_PTRS("three_nn", unknown, dist2, idx);
  if (m > 0 && !known) return fail(ISSM_E_NULL, "three_nn: known is NULL");
  return launched(launch_three_nn(b, n, m, unknown, known, dist2, idx, (hipStream_t)stream), "three_nn");
}

int issm_pn2_three_interpolate(int32_t b, int32_t c, int32_t m, int32_t n, const float* points, const int32_t* idx,
                               const float* weight, float* out, void* stream) {
  PN2_SIZES("three_interpolate", b, c, m, n);
  if ((int64_t)b * c * n == 0) return ISSM_OK;
  if (m == 0) return fail(ISSM_E_SHAPE, "three_interpolate: no points to index");
  PN2_PTRS("three_interpolate", points, idx, weight, out);
  return launched(launch_three_interpolate(b, c, m, n, points, idx, weight, out, (hipStream_t)stream), "three_interpolate");
}

int issm_pn2_three_interpolate_grad(int32_t b, int32_t c, int32_t n, int32_t m, const float* grad_out, const int32_t* idx,
                                    const float* weight, float* grad_points, void* stream) {
  PN2_SIZES("three_interpolate_grad", b, c, n, m);
  if ((int64_t)b * c * n == 0) return ISSM_OK;
  if (m == 0) return fail(ISSM_E_SHAPE, "three_interpolate_grad: no points to index");
  PN2_PTRS("three_interpolate_grad", grad_out, idx, weight, grad_points);
  return launched(launch_three_interpolate_grad(b, c, n, m, grad_out, idx, weight, grad_points, (hipStream_t)stream),
                  "three_interpolate_grad");
}

int64_t issm_pn2_three_interpolate_grad_rows_workspace(int32_t b, int32_t n, int32_t m) {
  return b < 0 || n < 0 || m < 0 ? 0 : (int64_t)sizeof(int) * interp_rows_grad_ints(b, n, m);
}

int issm_pn2_three_interpolate_grad_rows(int32_t b, int32_t c, int32_t n, int32_t m, const float* grad_out, const int32_t* idx,
                                         const float* weight, void* workspace, float* grad_points, void* stream) {
  PN2_SIZES("three_interpolate_grad_rows", b, c, n, m);
  if ((int64_t)b * c * n == 0) return ISSM_OK;
  if (m == 0) return fail(ISSM_E_SHAPE, "three_interpolate_grad_rows: no points to index");
  if (n > ISSM_PN2_ROW_POINTS || m > ISSM_PN2_ROW_POINTS || b > 65535 || (int64_t)b * c > 0x7fffffff / 1024)
    return fail(ISSM_E_UNSUPPORTED, "three_interpolate_grad_rows: n = %d or m = %d > %d, or too many rows", n, m, ISSM_PN2_ROW_POINTS);
  PN2_PTRS("three_interpolate_grad_rows", grad_out, idx, weight, workspace, grad_points);
  if ((uintptr_t)workspace & 7) return fail(ISSM_E_STRIDE, "three_interpolate_grad_rows: workspace is not aligned to 8 bytes");
  return launched(launch_interp_rows_grad(b, c, n, m, grad_out, idx, weight, (int*)workspace, grad_points, (hipStream_t)stream),
                  "three_interpolate_grad_rows");
}

int issm_pn2_group_points_grad_cl(int32_t b, int32_t c, int32_t n, int32_t npoints, int32_t nsample, const float* grad_out,
                                  const int32_t* idx, float* grad_points_cl, void* stream) {
  PN2_SIZES("group_points_grad_cl", b, c, n, npoints, nsample);
  if ((int64_t)b * c * npoints * nsample == 0) return ISSM_OK;
  if (n == 0) return fail(ISSM_E_SHAPE, "group_points_grad_cl: no points to index");
  if ((int64_t)npoints * nsample > 0x7fffffff || b > 65535)
    return fail(ISSM_E_UNSUPPORTED, "group_points_grad_cl: too many indices per sample or batch > 65535");
  PN2_PTRS("group_points_grad_cl", grad_out, idx, grad_points_cl);
  return launched(launch_scatter_channel_last(false, b, c, n, npoints * nsample, grad_out, idx, nullptr, grad_points_cl,
                                              (hipStream_t)stream), "group_points_grad_cl");
}

int issm_pn2_three_interpolate_grad_cl(int32_t b, int32_t c, int32_t n, int32_t m, const float* grad_out,
                                       const int32_t* idx, const float* weight, float* grad_points_cl, void* stream) {
  PN2_SIZES("three_interpolate_grad_cl", b, c, n, m);
  if ((int64_t)b * c * n == 0) return ISSM_OK;
  if (m == 0) return fail(ISSM_E_SHAPE, "three_interpolate_grad_cl: no points to index");
  if (b > 65535) return fail(ISSM_E_UNSUPPORTED, "three_interpolate_grad_cl: batch %d > 65535", b);
  PN2_PTRS("three_interpolate_grad_cl", grad_out, idx, weight, grad_points_cl);
  return launched(launch_scatter_channel_last(true, b, c, m, n, grad_out, idx, weight, grad_points_cl, (hipStream_t)stream),
                  "three_interpolate_grad_cl");
}

}  // extern "C"
