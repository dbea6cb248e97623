// Host side of the operators on PyTorch tensors: checks, argument blocks, output and workspace allocation and the autograd
// nodes around the entry points of libissm_hip.so.  One call of the scan takes some thirty tensor descriptors, a dozen
// allocations and an autograd node in each direction; issued from Python that is 100 - 300 us of host time for kernels
// that take 30 - 100 us at a single scene's size, and a decoder layer (four projections, the core, a norm) ran at the pace
// of the interpreter.  Here the same sequence costs the tensor library's own calls only.  All arithmetic is in the HIP
// kernels (and, for the layer's four projections, in the tensor library's matrix products).
#include <Python.h>

#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/extension.h>

#include <numeric>

#include "../../include/issm.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------------------------------------------- helpers
void check(int rc, const char* what) {
  if (rc != 0)
    throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(rc) + "): " + issm_last_error());
}

// Argument errors keep the exception types a Python implementation raises (called with the interpreter lock held).
[[noreturn]] void raise_py(PyObject* type, const std::string& msg) {
  PyErr_SetString(type, msg.c_str());
  throw py::error_already_set();
}
void require(bool ok, const char* msg) {
  if (!ok) raise_py(PyExc_AssertionError, msg);
}
void require_gpu(const Tensor& t, const char* name) {
  if (!t.is_cuda())
    raise_py(PyExc_RuntimeError, std::string(name) + " must live on a HIP device: the ISSM operator has no CPU path");
}
// The kernels take addresses: an operand on the host or on another device is refused before its address is used.
void require_beside(const Tensor& x, std::initializer_list<const Tensor*> operands) {
  for (const Tensor* t : operands)
    if (t->defined() && t->device() != x.device())
      raise_py(PyExc_RuntimeError, "all operands must be on " + x.device().str() + ", one is on " + t->device().str());
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool is_kernel_type(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
at::ScalarType kernel_type(at::ScalarType t) { return is_kernel_type(t) ? t : at::kFloat; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? ISSM_BF16 : ISSM_F32; }

Tensor cast(const Tensor& t, at::ScalarType type) { return !t.defined() || t.scalar_type() == type ? t : t.to(type); }
Tensor io_cast(const Tensor& t, at::ScalarType type) {
  if (!t.defined()) return t;
  Tensor r = cast(t, type);
  return r.stride(-1) == 1 ? r : r.contiguous();
}
Tensor f32c(const Tensor& t) { return t.defined() ? cast(t, at::kFloat).contiguous() : t; }
Tensor fresh(at::IntArrayRef sizes, const Tensor& like, at::ScalarType type) {
  return at::empty(sizes, like.options().dtype(type));
}
template <class T = void>
T* data(const Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }

issm_tensor desc(const Tensor& t) {
  issm_tensor d{};
  if (t.defined()) {
    TORCH_CHECK(t.dim() == 4 && t.stride(-1) == 1, "innermost dimension must be contiguous");
    d.ptr = t.data_ptr();
    for (int i = 0; i < 3; ++i) d.stride[i] = t.stride(i);
  }
  return d;
}

// What a backward pass needs to know of an input it does not read: its type and sizes.  (Such inputs are not saved: they may
// be changed in place between forward and backward, and need not be kept alive.)
struct Kind {
  at::ScalarType type = at::kFloat;
  at::DimVector sizes;
  Kind() = default;
  explicit Kind(const Tensor& t) {
    if (!t.defined()) return;
    type = t.scalar_type();
    sizes = at::DimVector(t.sizes());
  }
};
// A node's own record, beside its saved tensors
template <class T>
void keep(AutogradContext* ctx, c10::intrusive_ptr<T> record) { ctx->saved_data["record"] = c10::IValue::make_capsule(std::move(record)); }
template <class T>
c10::intrusive_ptr<T> kept(AutogradContext* ctx) { return c10::static_intrusive_pointer_cast<T>(ctx->saved_data["record"].toCapsule()); }

typedef c10::optional<Tensor> MaybeTensor;   // an absent input of a node: it takes no undefined tensors

Tensor opt(const MaybeTensor& t) { return t.has_value() ? *t : Tensor(); }

// ------------------------------------------------------------------------------------------------------------------- scan
// Kernel-ready operands of one call (1 or 2 directions).
struct Scan {
  int ndir = 1;
  Tensor x[2], dt, A, B[2], C[2], D, z[2], dt_bias, h0, seq;
  bool softplus = false;
  double lo = 0, hi = 0;

  static Scan make(int ndir, const Tensor (&x)[2], const Tensor& dt, const Tensor& A, const Tensor (&B)[2], const Tensor (&C)[2],
                   const Tensor& D, const Tensor (&z)[2], const Tensor& dt_bias, const Tensor& h0, const Tensor& seq,
                   bool softplus, double lo, double hi) {
    Scan s;
    s.ndir = ndir;
    const at::ScalarType io = kernel_type(x[0].scalar_type());
    for (int i = 0; i < ndir; ++i) {
      s.x[i] = io_cast(x[i], io);
      s.B[i] = io_cast(B[i], io);
      s.C[i] = io_cast(C[i], io);
      s.z[i] = io_cast(z[i], io);
    }
    s.dt = io_cast(dt, kernel_type(dt.scalar_type()));
    s.A = f32c(A);
    s.D = f32c(D);
    s.dt_bias = f32c(dt_bias);
    if (h0.defined()) s.h0 = io_cast(h0, kernel_type(h0.scalar_type()));
    if (seq.defined()) s.seq = cast(seq, at::kInt).contiguous();
    s.softplus = softplus;
    s.lo = lo;
    s.hi = hi;
    return s;
  }

  issm_scan_args args() const {
    issm_scan_args a{};
    a.dims.batch = (int)x[0].size(0);
    a.dims.seqlen = (int)x[0].size(1);
    a.dims.nheads = (int)x[0].size(2);
    a.dims.headdim = (int)x[0].size(3);
    a.dims.ngroups = (int)B[0].size(2);
    a.dims.dstate = (int)B[0].size(3);
    a.dims.chunk_size = ISSM_CHUNK;
    a.dims.ndir = ndir;
    a.io_dtype = code(x[0].scalar_type());
    a.dt_dtype = code(dt.scalar_type());
    a.h0_dtype = h0.defined() ? code(h0.scalar_type()) : ISSM_F32;
    a.flags = (softplus ? ISSM_FLAG_DT_SOFTPLUS : 0u) | (D.defined() && D.dim() == 2 ? ISSM_FLAG_D_HAS_HDIM : 0u);
    if (seq.defined()) {
      a.flags |= ISSM_FLAG_SEQ_IDX;
      a.seq_idx = data<const int32_t>(seq);
      a.seq_idx_stride[0] = seq.stride(0);
      a.seq_idx_stride[1] = seq.stride(1);
    }
    a.dt_min = (float)lo;
    a.dt_max = (float)std::min(hi, 3.0e38);
    for (int i = 0; i < ndir; ++i) {
      a.x[i] = desc(x[i]);
      a.Bm[i] = desc(B[i]);
      a.Cm[i] = desc(C[i]);
      a.z[i] = desc(z[i]);
    }
    a.dt = desc(dt);
    a.A = data<const float>(A);
    a.D = data<const float>(D);
    a.dt_bias = data<const float>(dt_bias);
    a.h0 = desc(h0);
    a.stream = stream_of(x[0]);
    return a;
  }

  struct Out {
    Tensor y[2], last[2], ws;
  };
  Out forward(bool want_last) const {
    issm_scan_args a = args();
    Out o;
    const auto& s = x[0].sizes();
    for (int i = 0; i < ndir; ++i) {
      o.y[i] = fresh(s, x[0], x[0].scalar_type());
      a.out[i] = desc(o.y[i]);
      if (want_last) {
        o.last[i] = fresh({s[0], s[2], s[3], B[0].size(3)}, x[0], at::kFloat);
        a.final_states[i] = data<float>(o.last[i]);
      }
    }
    size_t n = 0;
    check(issm_fwd_workspace_bytes(&a, &n), "workspace query");
    o.ws = fresh({(int64_t)std::max<size_t>(n, 256)}, x[0], at::kByte);
    a.workspace = data(o.ws);
    a.workspace_bytes = (size_t)o.ws.numel();
    check(issm_scan_fwd(&a), "issm_scan_fwd");
    return o;
  }

  struct Grad {
    Tensor dx[2], ddt, dA, dB[2], dC[2], dD, dz[2], dbias, dh0;
  };
  // dy: one per direction; dlast may be undefined (no gradient reaches the final states)
  Grad backward(const Tensor& ws_fwd, const Tensor (&dy_)[2], const Tensor (&dlast_)[2]) const {
    issm_scan_args a = args();
    const at::ScalarType io = x[0].scalar_type();
    a.saved = data(ws_fwd);
    Grad g;
    Tensor dy[2], dlast[2];
    for (int i = 0; i < ndir; ++i) {
      dy[i] = dy_[i].defined() ? io_cast(dy_[i], io) : at::zeros(x[i].sizes(), x[i].options());
      dlast[i] = f32c(dlast_[i]);
      g.dx[i] = fresh(x[i].sizes(), x[i], io);
      g.dB[i] = fresh(B[i].sizes(), x[i], io);
      g.dC[i] = fresh(C[i].sizes(), x[i], io);
      if (z[i].defined()) g.dz[i] = fresh(x[i].sizes(), x[i], io);
      a.dout[i] = desc(dy[i]);
      a.dfinal[i] = data<const float>(dlast[i]);
      a.dx[i] = desc(g.dx[i]);
      a.dB[i] = desc(g.dB[i]);
      a.dC[i] = desc(g.dC[i]);
      a.dz[i] = desc(g.dz[i]);
    }
    g.ddt = fresh(dt.sizes(), x[0], dt.scalar_type());
    g.dA = fresh(A.sizes(), x[0], at::kFloat);
    if (D.defined()) g.dD = fresh(D.sizes(), x[0], at::kFloat);
    if (dt_bias.defined()) g.dbias = fresh(dt_bias.sizes(), x[0], at::kFloat);
    g.dh0 = fresh({x[0].size(0), x[0].size(2), x[0].size(3), B[0].size(3)}, x[0], at::kFloat);
    a.ddt = desc(g.ddt);
    a.dA = data<float>(g.dA);
    a.dD = data<float>(g.dD);
    a.ddt_bias = data<float>(g.dbias);
    a.dh0 = data<float>(g.dh0);
    size_t n = 0;
    check(issm_bwd_workspace_bytes(&a, &n), "workspace query");
    Tensor ws = fresh({(int64_t)std::max<size_t>(n, 256)}, x[0], at::kByte);
    a.bwd_workspace = data(ws);
    a.bwd_workspace_bytes = (size_t)ws.numel();
    check(issm_scan_bwd(&a), "issm_scan_bwd");
    return g;
  }

  static constexpr int NSAVED = 14;
  void push(variable_list& v) const {
    for (const Tensor& t : {x[0], x[1], dt, A, B[0], B[1], C[0], C[1], D, z[0], z[1], dt_bias, h0, seq}) v.push_back(t);
  }
  static Scan pop(const variable_list& v, size_t at, int ndir, bool softplus, double lo, double hi) {
    Scan s;
    s.ndir = ndir;
    Tensor* to[NSAVED] = {&s.x[0], &s.x[1], &s.dt, &s.A, &s.B[0], &s.B[1], &s.C[0], &s.C[1], &s.D, &s.z[0], &s.z[1], &s.dt_bias,
                          &s.h0, &s.seq};
    for (int i = 0; i < NSAVED; ++i) *to[i] = v[at + i];
    s.softplus = softplus;
    s.lo = lo;
    s.hi = hi;
    return s;
  }
};

// Inputs 0 .. 11 of the node: x_f, x_b, dt, A, B_f, B_b, C_f, C_b, D, z, dt_bias, h0 (those of an absent direction undefined).
// The caller's own tensors are among the saved ones: reading them back is what makes the autograd engine raise when one of
// them was modified in place between forward and backward.
struct ScanFn : public Function<ScanFn> {
  static constexpr int NIN = 12;

  static variable_list forward(AutogradContext* ctx, const Tensor& x_f, const MaybeTensor& x_b_, const Tensor& dt, const Tensor& A,
                               const Tensor& B_f, const MaybeTensor& B_b_, const Tensor& C_f, const MaybeTensor& C_b_,
                               const MaybeTensor& D_, const MaybeTensor& z_, const MaybeTensor& dt_bias_, const MaybeTensor& h0_,
                               const MaybeTensor& seq_, bool softplus, double lo, double hi, bool want_last) {
    const c10::DeviceGuard guard(x_f.device());
    const Tensor x_b = opt(x_b_), B_b = opt(B_b_), C_b = opt(C_b_), D = opt(D_), z = opt(z_), dt_bias = opt(dt_bias_), h0 = opt(h0_),
                 seq = opt(seq_);
    const int ndir = x_b.defined() ? 2 : 1;
    const Tensor x[2] = {x_f, x_b}, B[2] = {B_f, B_b}, C[2] = {C_f, C_b}, zz[2] = {z, Tensor()};
    const Scan s = Scan::make(ndir, x, dt, A, B, C, D, zz, dt_bias, h0, seq, softplus, lo, hi);
    Scan::Out o = s.forward(want_last);
    ctx->set_materialize_grads(false);
    variable_list saved{x_f, x_b, dt, A, B_f, B_b, C_f, C_b, D, z, dt_bias, h0};
    s.push(saved);
    saved.push_back(o.ws);
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["ndir"] = (int64_t)ndir;
    ctx->saved_data["softplus"] = softplus;
    ctx->saved_data["lo"] = lo;
    ctx->saved_data["hi"] = hi;
    ctx->saved_data["last"] = want_last;
    variable_list out;
    for (int i = 0; i < ndir; ++i) out.push_back(cast(o.y[i], x[i].scalar_type()));
    if (want_last)
      for (int i = 0; i < ndir; ++i) out.push_back(o.last[i]);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list v = ctx->get_saved_variables();
    const int ndir = (int)ctx->saved_data["ndir"].toInt();
    const bool last = ctx->saved_data["last"].toBool();
    const Scan s = Scan::pop(v, NIN, ndir, ctx->saved_data["softplus"].toBool(), ctx->saved_data["lo"].toDouble(),
                             ctx->saved_data["hi"].toDouble());
    const c10::DeviceGuard guard(s.x[0].device());
    Tensor dy[2], dlast[2];
    for (int i = 0; i < ndir; ++i) {
      dy[i] = grads[i];
      if (last) dlast[i] = grads[ndir + i];
    }
    Scan::Grad g = s.backward(v[NIN + Scan::NSAVED], dy, dlast);
    const Tensor all[NIN] = {g.dx[0], g.dx[1], g.ddt, g.dA, g.dB[0], g.dB[1], g.dC[0], g.dC[1], g.dD, g.dz[0], g.dbias, g.dh0};
    variable_list out(NIN + 5);
    for (int i = 0; i < NIN; ++i)
      if (v[i].defined() && all[i].defined()) out[i] = cast(all[i], v[i].scalar_type());
    return out;
  }
};

std::string shape_text(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + ")";
}

// shape rules of issm_combined.py:58-83
void check_scan(const Tensor* x, const Tensor& dt, const Tensor& A, const Tensor* B, const Tensor* C, int ndir, const Tensor& D,
                const Tensor& z, const Tensor& dt_bias, const Tensor& h0, const Tensor& seq) {
  require_gpu(x[0], "x");
  for (int i = 0; i < ndir; ++i) require_beside(x[0], {&x[i], &B[i], &C[i]});
  require_beside(x[0], {&dt, &A, &D, &z, &dt_bias, &h0, &seq});
  if (x[0].dim() != 4) raise_py(PyExc_ValueError, "x must be (batch, seqlen, nheads, headdim), got " + shape_text(x[0]));
  if (B[0].dim() != 4) raise_py(PyExc_ValueError, "B must be (batch, seqlen, ngroups, dstate), got " + shape_text(B[0]));
  const int64_t b = x[0].size(0), l = x[0].size(1), h = x[0].size(2), p = x[0].size(3), g = B[0].size(2), n = B[0].size(3);
  require(g > 0 && h % g == 0, "nheads must be divisible by ngroups");
  for (int i = 0; i < ndir; ++i) {
    require(x[i].sizes() == at::IntArrayRef({b, l, h, p}), "x must be (batch, seqlen, nheads, headdim)");
    require(B[i].sizes() == at::IntArrayRef({b, l, g, n}), "B must be (batch, seqlen, ngroups, dstate)");
    require(C[i].sizes() == B[i].sizes(), "C must have B's shape");
  }
  require(dt.sizes() == at::IntArrayRef({b, l, h, n}), "dt must be (batch, seqlen, nheads, dstate)");
  require(A.sizes() == at::IntArrayRef({h, n}), "A must be (nheads, dstate)");
  if (z.defined()) require(z.sizes() == x[0].sizes(), "z must have x's shape");
  if (D.defined())
    require(D.sizes() == at::IntArrayRef({h, p}) || D.sizes() == at::IntArrayRef({h}), "D must be (nheads,) or (nheads, headdim)");
  if (dt_bias.defined()) require(dt_bias.sizes() == at::IntArrayRef({h, n}), "dt_bias must be (nheads, dstate)");
  if (h0.defined()) require(h0.sizes() == at::IntArrayRef({b, h, p, n}), "initial_states must be (batch, nheads, headdim, dstate)");
  if (seq.defined()) require(seq.sizes() == at::IntArrayRef({b, l}), "seq_idx must be (batch, seqlen)");
}

std::vector<Tensor> scan(const Tensor& x, const Tensor& dt, const Tensor& A, const Tensor& B, const Tensor& C,
                         const MaybeTensor& D_, const MaybeTensor& z_, const MaybeTensor& dt_bias_,
                         const MaybeTensor& h0_, const MaybeTensor& seq_, bool softplus, double lo, double hi,
                         bool want_last) {
  const Tensor D = opt(D_), z = opt(z_), dt_bias = opt(dt_bias_), h0 = opt(h0_), seq = opt(seq_);
  check_scan(&x, dt, A, &B, &C, 1, D, z, dt_bias, h0, seq);
  py::gil_scoped_release release;
  return ScanFn::apply(x, MaybeTensor(), dt, A, B, MaybeTensor(), C, MaybeTensor(), D_, z_, dt_bias_, h0_, seq_, softplus, lo, hi,
                       want_last);
}

std::vector<Tensor> biscan(const Tensor& x_f, const Tensor& x_b, const Tensor& dt, const Tensor& A, const Tensor& B_f,
                           const Tensor& B_b, const Tensor& C_f, const Tensor& C_b, const MaybeTensor& D_,
                           const MaybeTensor& dt_bias_, const MaybeTensor& h0_, bool softplus, double lo,
                           double hi) {
  const Tensor D = opt(D_), dt_bias = opt(dt_bias_), h0 = opt(h0_), none;
  const Tensor x[2] = {x_f, x_b}, B[2] = {B_f, B_b}, C[2] = {C_f, C_b};
  check_scan(x, dt, A, B, C, 2, D, none, dt_bias, h0, none);
  py::gil_scoped_release release;
  return ScanFn::apply(x_f, MaybeTensor(x_b), dt, A, B_f, MaybeTensor(B_b), C_f, MaybeTensor(C_b), D_, MaybeTensor(), dt_bias_, h0_,
                       MaybeTensor(), softplus, lo, hi, true);
}

// The checked argument block of a call, for callers of the C ABI from Python (stage entry points, preallocated buffers), and
// the tensors it points into.
std::pair<py::bytes, std::vector<Tensor>> scan_args(const Tensor& x_f, const MaybeTensor& x_b, const Tensor& dt, const Tensor& A,
                                                    const Tensor& B_f, const MaybeTensor& B_b, const Tensor& C_f,
                                                    const MaybeTensor& C_b, const MaybeTensor& D, const MaybeTensor& z_f,
                                                    const MaybeTensor& z_b, const MaybeTensor& dt_bias, const MaybeTensor& h0,
                                                    const MaybeTensor& seq, bool softplus, double lo, double hi) {
  const int ndir = x_b.has_value() ? 2 : 1;
  const Tensor x[2] = {x_f, opt(x_b)}, B[2] = {B_f, opt(B_b)}, C[2] = {C_f, opt(C_b)}, z[2] = {opt(z_f), opt(z_b)};
  for (int i = 0; i < ndir; ++i) check_scan(x, dt, A, B, C, ndir, opt(D), z[i], opt(dt_bias), opt(h0), opt(seq));
  const at::NoGradGuard no_grad;
  const Scan s = Scan::make(ndir, x, dt, A, B, C, opt(D), z, opt(dt_bias), opt(h0), opt(seq), softplus, lo, hi);
  const issm_scan_args a = s.args();
  std::vector<Tensor> used;
  s.push(used);
  return {py::bytes((const char*)&a, sizeof a), used};
}

// ------------------------------------------------------------------------------------------------------------- gated norm
Tensor as_rows(const Tensor& t) {
  Tensor r = t.reshape({-1, t.size(-1)});
  return r.stride(-1) == 1 ? r : r.contiguous();
}

issm_norm_args norm_args(const Tensor& x, const Tensor& z, const Tensor& w, const Tensor& bias, double eps, int64_t group,
                         bool before_gate, bool layer_norm) {
  issm_norm_args a{};
  a.rows = x.size(0);
  a.ncols = (int)x.size(1);
  a.group_size = (int)group;
  a.dtype = code(x.scalar_type());
  a.weight_dtype = code(w.scalar_type());
  a.norm_before_gate = before_gate;
  a.eps = (float)eps;
  a.x = data(x);
  a.w = data(w);
  a.x_row_stride = x.stride(0);
  if (z.defined()) {
    a.z = data(z);
    a.z_row_stride = z.stride(0);
  }
  a.bias = data(bias);
  a.layer_norm = layer_norm;
  a.stream = stream_of(x);
  return a;
}

struct NormFn : public Function<NormFn> {
  struct Record : torch::CustomClassHolder {
    Kind x, weight, bias, z;
    double eps;
    int64_t group;
    bool before_gate, rms;
  };

  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const MaybeTensor& bias_, const MaybeTensor& z_,
                        double eps, int64_t group, bool before_gate, bool rms) {
    const c10::DeviceGuard guard(x.device());
    const Tensor bias = opt(bias_), z = opt(z_);
    const at::ScalarType k = kernel_type(x.scalar_type());
    Tensor x2 = as_rows(cast(x, k)), z2, w = weight, b;
    if (z.defined()) z2 = as_rows(cast(z, k));
    if (!is_kernel_type(w.scalar_type())) w = w.to(at::kFloat);
    if (bias.defined()) {
      // The kernels read weight and bias in one dtype, the reference's widen each to fp32 on its own
      // (layernorm_gated.py:77-80): where the two differ both go to fp32, so that neither is rounded.
      if (bias.scalar_type() != w.scalar_type()) w = w.to(at::kFloat);
      b = cast(bias, w.scalar_type()).contiguous();
    }
    w = w.contiguous();
    const int64_t groups = group ? x2.size(1) / group : 1;
    Tensor y = fresh(x2.sizes(), x2, k), stats = fresh({2, groups * x2.size(0)}, x2, at::kFloat);
    issm_norm_args a = norm_args(x2, z2, w, b, eps, group, before_gate, !rms);
    a.y = data(y);
    a.y_row_stride = y.stride(0);
    a.rstd = data<float>(stats);
    if (!rms) a.mean = data<float>(stats) + stats.size(1);
    check(issm_gated_rmsnorm_fwd(&a), "issm_gated_rmsnorm_fwd");
    ctx->save_for_backward({x2, z2, w, b, stats});   // (x2, z2, w, b: the inputs themselves where the kernels read those)
    auto r = c10::make_intrusive<Record>();
    r->x = Kind(x);
    r->weight = Kind(weight);
    r->bias = Kind(bias);
    r->z = Kind(z);
    r->eps = eps;
    r->group = group;
    r->before_gate = before_gate;
    r->rms = rms;
    keep(ctx, std::move(r));
    return cast(y.view(x.sizes()), x.scalar_type());
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list v = ctx->get_saved_variables();
    const Tensor &x2 = v[0], &z2 = v[1], &w = v[2], &b = v[3], &stats = v[4];
    const auto in = kept<Record>(ctx);
    const c10::DeviceGuard guard(x2.device());
    const bool rms = in->rms;
    Tensor dy = as_rows(cast(grads[0], x2.scalar_type()));
    Tensor dx = fresh(x2.sizes(), x2, x2.scalar_type()), dz;
    if (z2.defined()) dz = fresh(z2.sizes(), z2, z2.scalar_type());
    const int64_t cols = x2.size(1), nb = issm_rmsnorm_bwd_blocks(x2.size(0)), np = b.defined() ? 2 : 1;
    // the gradients in the parameters' type where that is one that the kernels write
    const at::ScalarType wt = in->weight.type, type = is_kernel_type(wt) && (np == 1 || in->bias.type == wt) ? wt : at::kFloat;
    Tensor part = fresh({np, nb, cols}, x2, at::kFloat), dwb = fresh({np, cols}, x2, type);
    issm_norm_args a = norm_args(x2, z2, w, b, in->eps, in->group, in->before_gate, !rms);
    a.rstd = data<float>(stats);
    if (!rms) a.mean = data<float>(stats) + stats.size(1);
    a.dy = data(dy);
    a.dy_row_stride = dy.stride(0);
    a.dx = data(dx);
    a.dx_row_stride = dx.stride(0);
    if (dz.defined()) {
      a.dz = data(dz);
      a.dz_row_stride = dz.stride(0);
    }
    a.dw_partial = data<float>(part);
    a.dw = (float*)data(dwb);
    if (np == 2) {
      a.db_partial = data<float>(part) + nb * cols;
      a.db = (float*)(data<char>(dwb) + cols * dwb.element_size());
    }
    check(issm_gated_rmsnorm_bwd_as(&a, code(type)), "issm_gated_rmsnorm_bwd_as");
    variable_list out(8);
    out[0] = cast(dx.view(in->x.sizes), in->x.type);
    out[1] = cast(dwb.select(0, 0), in->weight.type);
    if (np == 2) out[2] = cast(dwb.select(0, 1), in->bias.type);
    if (dz.defined()) out[3] = cast(dz.view(in->z.sizes), in->z.type);
    return out;
  }
};

// group: 0 = the whole row
Tensor norm(const Tensor& x, const Tensor& weight, const MaybeTensor& bias_, const MaybeTensor& z_, double eps,
            int64_t group, bool before_gate, bool rms) {
  const Tensor bias = opt(bias_), z = opt(z_);
  require_gpu(x, "x");
  require_beside(x, {&weight, &bias, &z});
  if (z.defined()) require(z.sizes() == x.sizes(), "z must have x's shape");
  require(weight.dim() == 1 && weight.size(0) == x.size(-1), "weight must have one entry per column");
  if (bias.defined()) require(bias.dim() == 1 && bias.size(0) == x.size(-1), "bias must have one entry per column");
  require(group >= 0 && (group == 0 || x.size(-1) % group == 0), "group_size must divide the number of columns");
  py::gil_scoped_release release;
  return NormFn::apply(x, weight, bias_, z_, eps, group, before_gate, rms);
}

// ------------------------------------------------------------------------------------------------ projections of the layer
// y = x W^T for a (tokens, features) activation with thousands of tokens and a few hundred features (the four projections of
// the layer).  Forward and input gradient are the library products nn.Linear uses; the weight gradient dW = dy^T x contracts
// over the tokens, and as one product its (out x in) result makes only a few dozen tiles -- a fraction of the GPU, 54 us for
// 8192 x 288 -> 586 in bf16.  Here the tokens are cut into slices that run as one batched product and the slices' results are
// summed (24 us).
//
// The forward products of few tokens are issm_linear_fwd's: 4.6 us to issue where the library's take 19, and the kernels are no
// longer up to about this many multiply-adds, whatever the sizes (2048 x 288 -> 586: 5.0 us against 6.7; 448 -> 448 6.0 and 5.8).
constexpr double FEW_PRODUCTS = 3.5e8;
// With more tokens they are where a contraction of up to this many features is a few steps of its tiles (8192 tokens, issm_linear_fwd's and the
// library's in us: 96 -> 202 3.9 and 6.1, 288 -> 288 6.2 and 8.9, 288 -> 586 10.6 and 13.0, 384 -> 778 15.3 and 17.9, but 512 -> 512 12.9 and 10.0), and the
// gradients dx = dy W to as many features, from contractions of up to DX_CONTRACTION (2048 and 8192 tokens: 288 -> 288 5.1 and 6.2, 6.8 and 10.4; 586 -> 288
// 8.5 and 9.2, 11.6 and 16.3; 906 -> 448 11.5 and 10.5, 21.6 and 20.9; below 2048 tokens they are up to 1 us longer and 14 us sooner issued).
constexpr int64_t TILE_RESULTS = 384, DX_CONTRACTION = 640;
// (with results in whole multiples of 64 the library's larger tiles come out even, and are ahead where tokens fill the GPU with them many times:
// 16384 tokens, 256 -> 256 8.5 and 8.1, 288 -> 288 9.0 and 13.2; 32768, 320 -> 320 22.6 and 19.4, 288 -> 288 14.9 and 21.6; with other results the two
// meet at 65536 tokens: 288 -> 586 63.1 and 62.8, 352 -> 352 43.9 and 43.8)
bool tiled_tokens(int64_t tokens, int64_t results) { return tokens <= (results % 64 ? 32768 : 8192); }
// A layer without a gradient (scan_layer's chain) goes on taking them beyond that, for what the launches between them save, up to where it
// was ahead for 16 to 512 queries while its first products were linear.hip's (multiples of 32 up to 640 features).  Separate steps and chain now, both with
// tiles, in us, scenes of 1024 tokens and 256 queries unless said.  At the line, 64 features, 50 and 66 scenes 822 and 767, 1070 and 1004; 128, 32 587 and 568;
// 288, 6, 8 and 12 scenes 160 and 160, 205 and 203, 306 and 307, with 64 queries 97 and 95, 110 and 118, 145 and 157; 320, 3 and 4 103 and 103, 123 and 131, 16 queries
// and 2 scenes of 2048 81 and 79; 384, 2 and 3 90 and 94, 109 and 115; 512, 2 and 3 122 and 104, 145 and 127.  So it lies within 8 % of where either is ahead
// for 288 to 384 features, whose separate products are in tiles and in one launch; to both sides of those the chain stays ahead beyond it: 64, 287 scenes
// 4518 and 4284; 192, 34 716 and 680; 256, 19 458 and 439; 448, 5 195 and 189; 512, 4 171 and 170.
double chain_products(int64_t features) {
  return features <= 64 ? 5.5e8 : features == 320 ? 8.6e8 : features == 128 || features > 288 ? 1.1e9 : 1.4e9;
}
// The chain's convolutions and generation of dt, B and C are one launch up to this many threads of the generation, two queries each where their
// number is even: the first wave of a workgroup convolves while the others wait, and from 0.4 million threads on that costs more than the
// launch and what lies between the two.  8 heads, 64 features, 256 queries, scenes of 1024 tokens: 1, 2, 3, 5 and 12 47.6 us in two launches and 46.6 in one, 58.7
// and 57.8, 70.9 and 71.4, 98.8 and 99.6, 191 and 196; 288 features 57.3 and 55.2, 79.1 and 79.6, 95.0 and 94.1, 140 and 142, 305 and 320; 51 queries, 64
// features, 5, 8 and 31 scenes 65.6 and 63.6, 85.2 and 85.1, 237 and 241.
constexpr int64_t JOINED_THREADS = 400000;
// (tensors that stand for something else than their memory, under vmap, functionalization, a tensor subclass or a lazy
// negation, go to the library's product, which knows them)
bool own_memory(const Tensor& t) {
  using K = c10::DispatchKey;
  return t.has_storage() &&
         !t.key_set().has_any(c10::DispatchKeySet({K::Python, K::Functionalize, K::FuncTorchBatched, K::FuncTorchGradWrapper,
                                                   K::Batched, K::Negative, K::ZeroTensor}));
}
// a dispatch mode (one that counts or records operations, say) or a tracer sees the library's products, and none of the kernels here
bool watched() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}
// Whether this may be one of the two runs of a checkpointed segment, which are to give the same bits although the first of them (reentrant
// checkpointing) or the second records no gradient here.  A reentrant segment runs first in the forward of an autograd function --
// there, and in inference mode, forward-mode derivatives are off -- and again in a backward pass; one of the other kind with hooks on
// saved tensors both times.
bool runs_twice() {
  const c10::AutogradState& s = c10::AutogradState::get_tls_state();
  return (!s.get_fw_grad_mode() && !s.get_inference_mode()) || torch::autograd::get_current_graph_task_id() >= 0 ||
         (s.get_grad_mode() && !at::SavedTensorDefaultHooks::get_tls_state().stack.empty());
}
bool own_product(const Tensor& x, const Tensor& w) {
  if (watched() || !own_memory(x) || !own_memory(w)) return false;
  if (x.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16 || !x.is_cuda() || w.device() != x.device()) return false;
  if (w.dim() != 2 || x.dim() < 1 || x.size(-1) != w.size(1) || w.size(1) == 0 || w.size(1) % 32 || x.numel() == 0) return false;
  return x.is_contiguous() && w.is_contiguous() && (((uintptr_t)x.data_ptr() | (uintptr_t)w.data_ptr()) & 15) == 0;
}
bool few_tokens(const Tensor& x, const Tensor& w, double most = FEW_PRODUCTS) {
  return own_product(x, w) && (double)x.numel() * (double)w.size(0) <= most;
}
bool many_tokens(const Tensor& x, const Tensor& w) {
  return own_product(x, w) && w.size(0) >= 96 && w.size(1) <= TILE_RESULTS && tiled_tokens(x.numel() / x.size(-1), w.size(0));
}
// dx = dy W (issm_linear_dx)
bool own_dx(const Tensor& dy, const Tensor& w) {
  if (at::GradMode::is_enabled() || watched() || !own_memory(dy) || !own_memory(w)) return false;
  if (dy.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16 || !dy.is_cuda() || w.device() != dy.device()) return false;
  if (w.dim() != 2 || dy.dim() < 1 || dy.numel() == 0 || dy.size(-1) != w.size(0) || !dy.is_contiguous() || !w.is_contiguous()) return false;
  const int64_t tokens = dy.numel() / dy.size(-1);
  return w.size(0) % 2 == 0 && w.size(0) <= DX_CONTRACTION && w.size(1) % 2 == 0 && w.size(1) >= 96 && w.size(1) <= TILE_RESULTS && tokens >= 64 &&
         tiled_tokens(tokens, w.size(1)) && (((uintptr_t)dy.data_ptr() | (uintptr_t)w.data_ptr()) & 3) == 0;
}
// One or two products in a launch, `kernel` issm_linear_fwd (y = x w^T) or issm_linear_dx (y = x w)
struct Product {
  const Tensor *x, *w;
  Tensor y;
};
template <int N>
void launch_products(int (*kernel)(const issm_linear_args*), bool dx, Product (&p)[N]) {
  const c10::DeviceGuard guard(p[0].x->device());
  issm_linear_args a{};
  for (int i = 0; i < N; ++i) {
    const Tensor &x = *p[i].x, &w = *p[i].w;
    at::DimVector sizes(x.sizes());
    sizes.back() = w.size(dx ? 1 : 0);
    p[i].y = fresh(sizes, x, at::kBFloat16);
    a.job[i] = issm_linear_job{data(x), data(w), data(p[i].y), x.numel() / x.size(-1), (int32_t)x.size(-1), (int32_t)sizes.back(), 0};
  }
  a.njobs = N;
  a.dtype = ISSM_BF16;
  a.stream = stream_of(*p[0].x);
  check(kernel(&a), dx ? "issm_linear_dx" : "issm_linear_fwd");
}
Tensor linear_own(const Tensor& x, const Tensor& w) {
  Product p[1] = {{&x, &w, {}}};
  launch_products(&issm_linear_fwd, false, p);
  return p[0].y;
}
Tensor linear_dx(const Tensor& dy, const Tensor& w) {
  Product p[1] = {{&dy, &w, {}}};
  launch_products(&issm_linear_dx, true, p);
  return p[0].y;
}

// Weight gradients with a small result are issm_linear_dw's: up to this many weights (586 x 288: 18.2 us against 24.8 at 8192
// tokens, 11.4 against 13.9 at 2048, 8.8 against 7.3 but a third of the host time at 256; 512 x 512 25.8 against 22.3).  A
// backward pass that is itself differentiated takes the library's products, which autograd knows.
constexpr int64_t DW_WEIGHTS = 200000;
bool narrow_result(const Tensor& x, const Tensor& dy) {
  return !at::GradMode::is_enabled() && !watched() && own_memory(x) && own_memory(dy) && x.is_cuda() && dy.device() == x.device() &&
         x.scalar_type() == at::kBFloat16 && dy.scalar_type() == at::kBFloat16 && x.is_contiguous() && dy.is_contiguous() &&
         x.size(0) > 0 && x.size(0) == dy.size(0) && x.size(0) < (1 << 30) && x.size(1) >= 6 && dy.size(1) >= 4 &&
         x.size(1) <= DW_WEIGHTS / dy.size(1);
}
// One or two of them in a launch
struct WeightGradient {
  Tensor x, dy, dw;
};
template <int N>
void launch_weight_gradients(WeightGradient (&g)[N]) {
  const c10::DeviceGuard guard(g[0].x.device());
  issm_linear_dw_args a[N];
  Tensor scratch[N];
  for (int i = 0; i < N; ++i) {
    const Tensor &x = g[i].x, &dy = g[i].dy;
    a[i] = issm_linear_dw_args{};
    a[i].tokens = x.size(0);
    a[i].in = (int32_t)x.size(1);
    a[i].out = (int32_t)dy.size(1);
    g[i].dw = fresh({dy.size(1), x.size(1)}, x, at::kBFloat16);
    scratch[i] = fresh({(int64_t)issm_linear_dw_scratch_bytes(a[i].tokens, a[i].in, a[i].out)}, x, at::kByte);
    a[i].dy = data(dy);
    a[i].x = data(x);
    a[i].dw = data(g[i].dw);
    a[i].dtype = ISSM_BF16;
    a[i].scratch = data(scratch[i]);
    a[i].scratch_bytes = (size_t)scratch[i].numel();
    a[i].stream = stream_of(x);
  }
  if constexpr (N == 2) check(issm_linear_dw_pair(&a[0], &a[1]), "issm_linear_dw_pair");
  else check(issm_linear_dw(&a[0]), "issm_linear_dw");
}
Tensor weight_gradient(const Tensor& x2, const Tensor& dy2) {
  if (narrow_result(x2, dy2)) {
    WeightGradient g[1] = {{x2, dy2, {}}};
    launch_weight_gradients(g);
    return g[0].dw;
  }
  const int64_t tokens = x2.size(0);
  int64_t slices = x2.scalar_type() == at::kBFloat16 ? 4 : 2;   // fastest of 2 .. 32 on MI355X at 2048 and 8192 tokens
  if (tokens < 1024 || tokens % slices) slices = 1;
  if (slices > 1)
    return at::bmm(dy2.view({slices, tokens / slices, -1}).transpose(1, 2), x2.view({slices, tokens / slices, -1})).sum(0);
  return at::mm(dy2.t(), x2);
}

bool own_linear(const Tensor& x, const Tensor& w) { return few_tokens(x, w) || many_tokens(x, w); }
struct LinearFn : public Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    ctx->save_for_backward({x, w});
    return own_linear(x, w) ? linear_own(x, w) : at::linear(x, w);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    // (whatever autocast says where backward() is called: the products below see operands of one type already)
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
    const variable_list v = ctx->get_saved_variables();
    const Tensor &x = v[0], &w = v[1];
    const Tensor dy = cast(grads[0], x.scalar_type());
    Tensor dx, dw;
    if (ctx->needs_input_grad(0)) dx = own_dx(dy, w) ? linear_dx(dy, w) : at::matmul(dy, w);
    if (ctx->needs_input_grad(1)) dw = weight_gradient(x.reshape({-1, x.size(-1)}), dy.reshape({-1, dy.size(-1)}));
    return {dx, dw};
  }
};

// The projections of keys and queries that stand beside each other in the layer, as one node: where both are products of the kernels here, forward, input
// and weight gradients take one launch for the two (and the weight gradients' sums another) instead of two each, the shorter one beside the other:
// 8 x 1024 keys and 8 x 256 queries, 288 features, us a pair: forward 15.1 -> 10.2, dx 16.6 -> 11.4, dW 19.5 -> 13.3 and its sums 9.1 -> 4.6.
// What a side saves is its own: a backward pass that wants the one neither looks at the other's tensors (which may have been changed in place) nor frees
// them, so that a second pass may want those.
struct PairRecord : torch::CustomClassHolder {
  torch::autograd::SavedVariable saved[2][2];   // of either side x, w
  void save(int side, const Tensor& x, const Tensor& w) {
    saved[side][0] = torch::autograd::SavedVariable(x, false);
    saved[side][1] = torch::autograd::SavedVariable(w, false);
  }
};
struct LinearPairFn : public Function<LinearPairFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x0, const Tensor& w0, const Tensor& x1, const Tensor& w1,
                               const c10::intrusive_ptr<PairRecord>& record) {
    keep(ctx, record);
    ctx->set_materialize_grads(false);   // an output that nothing was made of gives its weight no gradient
    if (own_linear(x0, w0) && own_linear(x1, w1) && x0.device() == x1.device()) {
      Product p[2] = {{&x0, &w0, {}}, {&x1, &w1, {}}};
      launch_products(&issm_linear_fwd, false, p);
      return {p[0].y, p[1].y};
    }
    return {own_linear(x0, w0) ? linear_own(x0, w0) : at::linear(x0, w0), own_linear(x1, w1) ? linear_own(x1, w1) : at::linear(x1, w1)};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
    const auto record = kept<PairRecord>(ctx);
    Tensor x[2], w[2], dy[2], out[4];
    bool want_x[2], want_w[2], want[2];
    for (int i = 0; i < 2; ++i) {
      want_x[i] = grads[i].defined() && ctx->needs_input_grad(2 * i);
      want_w[i] = grads[i].defined() && ctx->needs_input_grad(2 * i + 1);
      want[i] = want_x[i] || want_w[i];
      if (!want[i]) continue;
      x[i] = record->saved[i][0].unpack();
      w[i] = record->saved[i][1].unpack();
      dy[i] = cast(grads[i], x[i].scalar_type());
    }
    if (want_x[0] && want_x[1] && x[0].device() == x[1].device() && own_dx(dy[0], w[0]) && own_dx(dy[1], w[1])) {
      Product p[2] = {{&dy[0], &w[0], {}}, {&dy[1], &w[1], {}}};
      launch_products(&issm_linear_dx, true, p);
      out[0] = p[0].y;
      out[2] = p[1].y;
    } else {
      for (int i = 0; i < 2; ++i)
        if (want_x[i]) out[2 * i] = own_dx(dy[i], w[i]) ? linear_dx(dy[i], w[i]) : at::matmul(dy[i], w[i]);
    }
    WeightGradient g[2];
    for (int i = 0; i < 2; ++i)
      if (want_w[i]) g[i] = {x[i].reshape({-1, x[i].size(-1)}), dy[i].reshape({-1, dy[i].size(-1)}), {}};
    if (want_w[0] && want_w[1] && x[0].device() == x[1].device() && narrow_result(g[0].x, g[0].dy) && narrow_result(g[1].x, g[1].dy)) {
      launch_weight_gradients(g);
      out[1] = g[0].dw;
      out[3] = g[1].dw;
    } else {
      for (int i = 0; i < 2; ++i)
        if (want_w[i]) out[2 * i + 1] = weight_gradient(g[i].x, g[i].dy);
    }
    // (as a node's own saved tensors; what has been freed says so when it is asked for again)
    if (!torch::autograd::get_current_graph_task_keep_graph())
      for (int i = 0; i < 2; ++i)
        for (auto& s : record->saved[i])
          if (want[i]) s.reset_data();
    return {out[0], out[1], out[2], out[3], Tensor()};
  }
};

// under autocast the product runs in the autocast type; what is saved must be in that type too, or the backward would mix types
void autocast_types(std::initializer_list<Tensor*> operands) {
  if (!at::autocast::is_autocast_enabled(at::kCUDA)) return;
  const at::ScalarType type = at::autocast::get_autocast_dtype(at::kCUDA);
  for (Tensor* t : operands)
    if (t->scalar_type() != at::kDouble) *t = t->to(type);
}
Tensor linear_tokens(Tensor x, Tensor w) {
  autocast_types({&x, &w});
  const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
  return LinearFn::apply(x, w);
}
variable_list linear_pair(Tensor x0, Tensor w0, Tensor x1, Tensor w1) {
  // (a node's outputs all need a gradient or none)
  if ((x0.requires_grad() || w0.requires_grad()) != (x1.requires_grad() || w1.requires_grad())) return {linear_tokens(x0, w0), linear_tokens(x1, w1)};
  autocast_types({&x0, &w0, &x1, &w1});
  const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
  const auto record = c10::make_intrusive<PairRecord>();
  variable_list y = LinearPairFn::apply(x0, w0, x1, w1, record);
  if (y[0].requires_grad()) {
    record->save(0, x0, w0);
    record->save(1, x1, w1);
  }
  return y;
}

// ------------------------------------------------------------------------------- the chain between a layer's projections
// (B, R, C) -> (B, C, R): alpha * (in0 + in1) in `type`; in1 may be undefined (issm_transpose_states)
struct Turn {   // (its tensors kept while the arguments point to them)
  Tensor in0, in1, out;
  issm_transpose_args a{};
  Turn(const Tensor& in0_, const Tensor& in1_, double alpha, at::ScalarType type);
};
Turn::Turn(const Tensor& in0_, const Tensor& in1_, double alpha, at::ScalarType type) {
  const at::ScalarType k = kernel_type(in0_.scalar_type());
  in0 = cast(in0_, k).contiguous();
  in1 = in1_.defined() ? cast(in1_, k).contiguous() : in1_;
  out = fresh({in0.size(0), in0.size(2), in0.size(1)}, in0, type);
  a.batch = (int)in0.size(0);
  a.rows = (int)in0.size(1);
  a.cols = (int)in0.size(2);
  a.in_dtype = code(k);
  a.out_dtype = code(type);
  a.in0 = data(in0);
  a.in1 = data(in1);
  a.out = data(out);
  a.alpha = (float)alpha;
  a.stream = stream_of(in0);
}
Tensor transpose_states(const Tensor& in0, const Tensor& in1, double alpha, at::ScalarType type) {
  const Turn t(in0, in1, alpha, type);
  check(issm_transpose_states(&t.a), "issm_transpose_states");
  return t.out;
}

constexpr int TAPS = 7;   // of the depthwise convolutions
constexpr int WIDTH = 16; // of the distance encoding

issm_dwconv_args conv_args(const Tensor& u) {
  issm_dwconv_args a{};
  a.batch = (int)u.size(0);
  a.seqlen = (int)u.size(1);
  a.channels = (int)u.size(2);
  a.nsets = 2;
  a.taps = TAPS;
  a.dtype = code(u.scalar_type());
  a.u = data(u);
  a.u_batch_stride = u.stride(0);
  a.u_token_stride = u.stride(1);
  a.chain = 1;   // key_conv_back reads key_conv's output
  a.stream = stream_of(u);
  return a;
}

issm_pgen_args pgen_args(const Tensor& dist, const float* W, int64_t H, int64_t G) {
  issm_pgen_args a{};
  a.tokens = dist.size(0) * dist.size(1);
  a.K = (int)dist.size(2);
  a.M = (int)dist.size(3);
  a.H = (int)H;
  a.G = (int)G;
  a.dtype = code(dist.scalar_type());
  a.has_back = 1;
  a.dist = data(dist);
  a.W = W;
  a.stream = stream_of(dist);
  return a;
}

// Depthwise conv + SiLU of both branches (the reversed-order branch convolves the forward-order branch's output,
// dest_module.py:530,534), generation of dt / B / C from the distance encoding, the bidirectional scan, the average of the two
// directions and the gated RMSNorm as one autograd node (dest_module.py:528-581): the entry points of libissm_hip.so back to
// back, and their backward passes chained by hand.
struct CoreFn : public Function<CoreFn> {
  // the small parameters, in the order of their places in the flat fp32 buffer
  enum { CW_F, CW_B, CB_F, CB_B, DT_W, BC_W, DT_BIAS, A_LOG, D_, NSMALL };
  // (the kernels address the parameters by the layer's sizes: none may be smaller than its place)
  static void check_sizes(int64_t features, const Tensor& conv_w_f, const Tensor& conv_w_b, const Tensor& conv_b_f,
                          const Tensor& conv_b_b, const Tensor& dt_w, const Tensor& bc_w, const Tensor& dt_bias, const Tensor& A_log,
                          const Tensor& D, const Tensor& norm_w, int64_t di, int64_t H, int64_t G) {
    const int64_t Cc = di + 2 * G;
    auto has = [](const Tensor& t, int64_t n, const char* name) {
      TORCH_CHECK(t.numel() == n, name, " must have ", n, " entries, got ", t.numel());
    };
    TORCH_CHECK(features == di + Cc + H, "key_proj must give ", di + Cc + H, " features, got ", features);
    has(conv_w_f, Cc * TAPS, "key_conv.weight");
    has(conv_w_b, Cc * TAPS, "key_conv_back.weight");
    has(conv_b_f, Cc, "key_conv.bias");
    has(conv_b_b, Cc, "key_conv_back.bias");
    has(dt_w, H * WIDTH, "dt_proj.weight");
    has(bc_w, 2 * G * WIDTH, "bc_proj.weight");
    has(dt_bias, H, "dt_bias");
    has(A_log, H, "A_log");
    has(D, D.dim() == 1 ? H : di, "D");
    has(norm_w, di, "key_norm.weight");
  }
  // places of the arrays in the flat buffer; its length
  static int64_t offsets(const std::array<const Tensor*, NSMALL>& arrays, int64_t (&off)[NSMALL + 1]) {
    off[0] = 0;
    for (int i = 0; i < NSMALL; ++i) off[i + 1] = off[i] + arrays[i]->numel();
    return off[NSMALL];
  }
  static void small_parameters(const std::array<const Tensor*, NSMALL>& arrays, int64_t K, float* flat, float* A, void* stream,
                               const issm_linear_args* with = nullptr, const issm_transpose_args* turn = nullptr) {   // with, turn: in their launch
    static_assert(NSMALL == ISSM_LAYER_ARRAYS, "one array per parameter");
    issm_layer_params_args a{};
    Tensor kept[NSMALL];
    for (int i = 0; i < NSMALL; ++i) {
      kept[i] = cast(*arrays[i], kernel_type(arrays[i]->scalar_type())).contiguous();
      a.src[i] = data(kept[i]);
      a.n[i] = (int32_t)kept[i].numel();
      a.dtype[i] = code(kept[i].scalar_type());
    }
    a.a_log = A_LOG;
    a.K = (int32_t)K;
    a.out = flat;
    a.A = A;
    a.stream = stream;
    check(with ? issm_layer_in(with, &a) : turn ? issm_layer_begin(&a, turn) : issm_layer_params(&a), "issm_layer_params");
  }

  // tensor inputs: zxbcdt, h0_lin, dist, weights, conv_w_f, conv_b_f, conv_w_b, conv_b_b, dt_w, bc_w, dt_bias, A_log, D, norm_w
  static constexpr int NIN = 14;
  struct Record : torch::CustomClassHolder {
    Kind in[NIN];
    int64_t H, G, di;
    double lo, hi, eps;
  };

  static variable_list forward(AutogradContext* ctx, const Tensor& zxbcdt, const Tensor& h0_lin, const Tensor& dist,
                               const MaybeTensor& weights_, const Tensor& conv_w_f, const Tensor& conv_b_f, const Tensor& conv_w_b,
                               const Tensor& conv_b_b, const Tensor& dt_w, const Tensor& bc_w, const Tensor& dt_bias,
                               const Tensor& A_log, const Tensor& D, const Tensor& norm_w, int64_t d_inner, int64_t nheads,
                               int64_t ngroups, double lo, double hi, double eps) {
    const c10::DeviceGuard guard(zxbcdt.device());
    const Tensor weights = opt(weights_);
    const int64_t Bsz = zxbcdt.size(0), Ln = zxbcdt.size(1), H = nheads, G = ngroups, di = d_inner, P = di / H, Cc = di + 2 * G,
                  K = dist.size(2);
    const at::ScalarType k = kernel_type(zxbcdt.scalar_type());
    check_sizes(zxbcdt.size(2), conv_w_f, conv_w_b, conv_b_f, conv_b_b, dt_w, bc_w, dt_bias, A_log, D, norm_w, di, H, G);
    Tensor zx = io_cast(zxbcdt, k);
    const Tensor z = zx.narrow(2, 0, di), xbc = zx.narrow(2, di, Cc);
    // all small parameters in one fp32 buffer, and A for all state columns; adjacent pieces form the stacked operands the
    // kernels take
    int64_t off[NSMALL + 1];
    const std::array<const Tensor*, NSMALL> arrays{&conv_w_f, &conv_w_b, &conv_b_f, &conv_b_b, &dt_w, &bc_w, &dt_bias, &A_log, &D};
    Tensor flat = fresh({offsets(arrays, off)}, zx, at::kFloat), A1 = fresh({H, K}, zx, at::kFloat);
    // (and the queries in the layout of the scan's initial states)
    const Turn states(h0_lin.reshape({Bsz, K, di}), Tensor(), 1.0, kernel_type(h0_lin.scalar_type()));
    small_parameters(arrays, K, data<float>(flat), data<float>(A1), stream_of(zx), nullptr, &states.a);
    float* const par = data<float>(flat);
    // 1. both depthwise convolutions + SiLU; the conv writes x and the B / C biases apart
    Tensor x = fresh({2, Bsz, Ln, H, P}, zx, k), tail = fresh({2, Bsz, Ln, 2 * G}, zx, k), pre = fresh({2, Bsz, Ln, Cc}, zx, k);
    {
      issm_dwconv_args a = conv_args(xbc);
      a.w = par;
      a.bias = par + off[CB_F];
      a.y = data(x);
      a.pre = data(pre);
      a.split = (int)di;
      a.y_tail = data(tail);
      check(issm_dwconv_silu_fwd(&a), "issm_dwconv_silu_fwd");
    }
    // 2. dt / B / C (and the reversed-order B / C) from the distance encoding
    const Tensor d = cast(dist, k).contiguous(), wt = f32c(weights);
    Tensor dt = fresh({Bsz, Ln, H, K}, zx, k), bc = fresh({4, Bsz, Ln, G, K}, zx, k), raw;
    {
      issm_pgen_args a = pgen_args(d, par + off[DT_W], H, G);
      a.tok = (const char*)data(zx) + (di + Cc) * zx.element_size();
      a.tok_stride = zx.stride(1);
      a.tok_add = par + off[DT_BIAS];
      a.tail = data(tail);
      a.dt = data(dt);
      void** to[4] = {&a.Bm, &a.Cm, &a.Bm_back, &a.Cm_back};
      for (int i = 0; i < 4; ++i) *to[i] = (char*)data(bc) + i * (bc.numel() / 4) * bc.element_size();
      if (wt.defined()) {
        raw = fresh(dt.sizes(), zx, k);
        a.weights = data<const float>(wt);
        a.dt_raw = data(raw);
      }
      check(issm_param_gen_fwd(&a), "issm_param_gen_fwd");
    }
    // 3. the bidirectional scan, queries as initial state
    const Tensor h0 = states.out.view({Bsz, H, P, K});
    const Tensor xs[2] = {x.select(0, 0), x.select(0, 1)}, Bs[2] = {bc.select(0, 0), bc.select(0, 2)},
                 Cs[2] = {bc.select(0, 1), bc.select(0, 3)}, none[2];
    const Scan s = Scan::make(2, xs, dt, A1, Bs, Cs, D.dim() == 1 ? flat.narrow(0, off[D_], H) : D, none, Tensor(), h0,
                              Tensor(), !wt.defined(), lo, hi);
    Scan::Out o = s.forward(true);
    // 4. gated RMSNorm (norm(x * silu(z))) of the two directions' average: the norm of s / 2 with eps is the norm of s with
    // 4 eps, so the sum goes in as it is and the halving never runs (nor its backward)
    const bool together = di % 4 == 0 && di <= 1024;   // in one launch with the average of the final states
    const Tensor key = together ? fresh({Bsz * Ln, di}, zx, k) : at::add(o.y[0], o.y[1]).view({Bsz * Ln, di});
    const Tensor z2 = z.as_strided({Bsz * Ln, di}, {zx.stride(1), 1});
    const Tensor nw = cast(norm_w, kernel_type(norm_w.scalar_type())).contiguous();
    Tensor key_n = fresh(key.sizes(), key, k), rstd = fresh({Bsz * Ln}, key, at::kFloat);
    const Turn final(o.last[0].view({Bsz, di, K}), o.last[1].view({Bsz, di, K}), 0.5, kernel_type(h0_lin.scalar_type()));
    {
      issm_norm_args a = norm_args(key, z2, nw, Tensor(), 4.0 * eps, 0, false, false);
      a.y = data(key_n);
      a.y_row_stride = key_n.stride(0);
      a.rstd = data<float>(rstd);
      if (together) {
        a.x = data(o.y[0]);
        check(issm_layer_behind(&a, data(o.y[1]), data(key), &final.a), "issm_layer_behind");
      } else {
        check(issm_gated_rmsnorm_fwd(&a), "issm_gated_rmsnorm_fwd");
        check(issm_transpose_states(&final.a), "issm_transpose_states");
      }
    }
    const Tensor last = final.out;
    variable_list saved{xbc, pre, flat, d, wt, raw, key, z2, nw, rstd, A1, o.ws};
    s.push(saved);
    ctx->save_for_backward(std::move(saved));
    auto r = c10::make_intrusive<Record>();
    const Tensor* ins[NIN] = {&zxbcdt, &h0_lin, &dist, &weights, &conv_w_f, &conv_b_f, &conv_w_b, &conv_b_b, &dt_w, &bc_w, &dt_bias,
                              &A_log, &D, &norm_w};
    for (int i = 0; i < NIN; ++i) r->in[i] = Kind(*ins[i]);
    r->H = H;
    r->G = G;
    r->di = di;
    r->lo = lo;
    r->hi = hi;
    r->eps = 4.0 * eps;
    keep(ctx, std::move(r));
    return {cast(key_n.view({Bsz, Ln, di}), zxbcdt.scalar_type()), cast(last, h0_lin.scalar_type())};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::DispatchKey::AutocastCUDA);
    const variable_list v = ctx->get_saved_variables();
    const Tensor &xbc = v[0], &pre = v[1], &flat = v[2], &d = v[3], &wt = v[4], &raw = v[5], &key = v[6], &z2 = v[7], &nw = v[8],
                 &rstd = v[9], &A1 = v[10], &ws = v[11];
    const auto r = kept<Record>(ctx);
    const Kind* in = r->in;
    const c10::DeviceGuard guard(key.device());
    const int64_t H = r->H, G = r->G, di = r->di, P = di / H, Cc = di + 2 * G, Bsz = d.size(0), Ln = d.size(1),
                  K = d.size(2), R0 = H + 2 * G, Wd = di + Cc + H;
    const Scan s = Scan::pop(v, 12, 2, !wt.defined(), r->lo, r->hi);
    const at::ScalarType k = key.scalar_type(), hdt = in[1].type;
    float* const par = data<float>(flat);
    const int64_t off_w = 2 * Cc * TAPS + 2 * Cc;
    // 4'. gated RMSNorm
    const Tensor dy = cast(grads[0], k).reshape({Bsz * Ln, di}).contiguous();
    Tensor dkey = fresh(key.sizes(), key, k);
    Tensor dzx = fresh({Bsz, Ln, Wd}, key, k);   // row of d zxbcdt: [dz | d xbc | d dt]; each producer writes its part
    const int64_t nb = issm_rmsnorm_bwd_blocks(Bsz * Ln);
    Tensor dwp = fresh({nb, di}, key, at::kFloat);
    {
      issm_norm_args a = norm_args(key, z2, nw, Tensor(), r->eps, 0, false, false);
      a.rstd = data<float>(rstd);
      a.dy = data(dy);
      a.dy_row_stride = dy.stride(0);
      a.dx = data(dkey);
      a.dx_row_stride = dkey.stride(0);
      a.dz = data(dzx);
      a.dz_row_stride = Wd;
      a.dw_partial = data<float>(dwp);
      check(issm_gated_rmsnorm_bwd_part(&a), "issm_gated_rmsnorm_bwd_part");
    }
    // 3'. the scan: both directions receive the gradient of their sum, and half of the averaged final states'
    const Tensor dyh = dkey.view({Bsz, Ln, H, P});
    const Tensor dfin = transpose_states(grads[1].reshape({Bsz, K, di}), Tensor(), 0.5, at::kFloat).view({Bsz, H, P, K});
    const Tensor dys[2] = {dyh, dyh}, dlast[2] = {dfin, dfin};
    const Scan::Grad g = s.backward(ws, dys, dlast);
    // 2'. parameter generation; the gradients of its biases go to the convolutions' backward and to dzx
    const int gen_rows = issm_param_gen_bwd_blocks(Bsz * Ln);
    Tensor ddist, dwpart = fresh({std::max(gen_rows, 1), R0, WIDTH + 1}, key, at::kFloat), dtail = fresh({2, Bsz, Ln, 2 * G}, key, k);
    if (ctx->needs_input_grad(2)) ddist = fresh(d.sizes(), d, k);
    {
      issm_pgen_args a = pgen_args(d, par + off_w, H, G);
      a.ddt = data(g.ddt);
      a.dBm = data(g.dB[0]);
      a.dCm = data(g.dC[0]);
      a.dBm_back = data(g.dB[1]);
      a.dCm_back = data(g.dC[1]);
      a.ddist = data(ddist);
      a.dw_partial = data<float>(dwpart);
      if (wt.defined()) {
        a.weights = data<const float>(wt);
        a.dt_raw = data(raw);
      }
      const issm_pgen_producers to{(char*)data(dzx) + (di + Cc) * dzx.element_size(), Wd, data(dtail)};
      check(issm_param_gen_bwd_part(&a, &to), "issm_param_gen_bwd_part");
    }
    // 1'. the convolutions: gradients of (x, b-bias, c-bias) per branch
    const int conv_rows = issm_dwconv_part_rows((int)Bsz, (int)Ln);
    Tensor part = fresh({std::max(conv_rows, 1), 2, 8, Cc}, key, at::kFloat);
    {
      issm_dwconv_args a = conv_args(xbc);
      a.w = par;
      a.pre = data(pre);
      a.split = (int)di;
      for (int i = 0; i < 2; ++i) {
        a.dy[i] = data(g.dx[i]);
        a.dy_tail[i] = (char*)data(dtail) + i * (dtail.numel() / 2) * dtail.element_size();
      }
      a.du = (char*)data(dzx) + di * dzx.element_size();
      a.du_batch_stride = Ln * Wd;
      a.du_token_stride = Wd;
      a.partial = data<float>(part);
      check(issm_dwconv_silu_bwd_part(&a), "issm_dwconv_silu_bwd_part");
    }
    // the sums of all the parts, inputs 4 .. 13, in the parameters' type when they share one, and the queries' gradient
    bool bf16 = true;
    for (int i = 4; i < NIN; ++i) bf16 = bf16 && in[i].type == at::kBFloat16;
    const std::vector<int64_t> n{Cc * TAPS, Cc, Cc * TAPS, Cc, H * WIDTH, 2 * G * WIDTH, H, H, g.dD.numel(), di};
    Tensor dh0 = fresh({Bsz, K, di}, key, kernel_type(hdt)),
           sums = fresh({std::accumulate(n.begin(), n.end(), (int64_t)0)}, key, bf16 ? at::kBFloat16 : at::kFloat);
    {
      issm_layer_grads_args a{};
      a.conv = data<const float>(part);
      a.gen = data<const float>(dwpart);
      a.norm = data<const float>(dwp);
      a.conv_rows = conv_rows;
      a.gen_rows = gen_rows;
      a.norm_rows = (int32_t)nb;
      a.C = (int32_t)Cc;
      a.H = (int32_t)H;
      a.G = (int32_t)G;
      a.d_inner = (int32_t)di;
      a.K = (int32_t)K;
      a.dA = data<const float>(g.dA);
      a.A = data<const float>(A1);
      a.dD = data<const float>(g.dD);
      a.nD = (int32_t)g.dD.numel();
      a.dtype = code(sums.scalar_type());
      a.out = data(sums);
      a.stream = stream_of(key);
      issm_transpose_args t{};
      t.batch = (int)Bsz;
      t.rows = (int)di;
      t.cols = (int)K;
      t.in_dtype = ISSM_F32;
      t.out_dtype = code(dh0.scalar_type());
      t.in0 = data(g.dh0);
      t.out = data(dh0);
      t.alpha = 1.0f;
      check(issm_layer_grads(&a, &t), "issm_layer_grads");
    }
    const std::vector<Tensor> pg = at::split_with_sizes(sums, n);
    variable_list out(NIN + 6);
    out[0] = cast(dzx, in[0].type);
    out[1] = cast(dh0, hdt);
    out[2] = cast(ddist, in[2].type);
    for (int i = 4; i < NIN; ++i) out[i] = cast(pg[i - 4], in[i].type).view(in[i].sizes);
    return out;
  }
};

// What lies between the input projections and the output projections (dest_module.py:528-581): zx (B, L, 2 d_inner + 2 G + H)
// from key_proj, h0 (B, K, d_inner) from query_proj -> the normalised key and the averaged final states.
void check_core(const Tensor& zx, const Tensor& h0, const Tensor& dist, const Tensor& weights, int64_t d_inner, int64_t nheads,
                int64_t ngroups, std::initializer_list<const Tensor*> parameters) {
  require_gpu(zx, "in_key");
  require_beside(zx, {&h0, &dist, &weights});
  require_beside(zx, parameters);
  require(nheads > 0 && ngroups > 0 && d_inner % nheads == 0 && nheads % ngroups == 0,
          "d_inner must be divisible by nheads, and nheads by ngroups");
  require(zx.dim() == 3 && h0.dim() == 3 && dist.dim() == 4, "in_key (B, L, D), in_query (B, K, D), dist (B, L, K, M)");
  require(dist.size(0) == zx.size(0) && dist.size(1) == zx.size(1) && h0.size(0) == zx.size(0) && dist.size(2) == h0.size(1) &&
              dist.size(3) == WIDTH, "dist must be (B, L, K, 16)");
  if (weights.defined()) require(weights.sizes() == dist.sizes().slice(0, 3), "mask must be (B, L, K)");
}

std::vector<Tensor> scan_core(const Tensor& zx, const Tensor& h0, const Tensor& dist, const MaybeTensor& weights_,
                              const Tensor& conv_w_f, const Tensor& conv_b_f, const Tensor& conv_w_b, const Tensor& conv_b_b,
                              const Tensor& dt_w, const Tensor& bc_w, const Tensor& dt_bias, const Tensor& A_log, const Tensor& D,
                              const Tensor& key_norm, double key_eps, int64_t d_inner, int64_t nheads, int64_t ngroups, double lo,
                              double hi) {
  check_core(zx, h0, dist, opt(weights_), d_inner, nheads, ngroups,
             {&conv_w_f, &conv_b_f, &conv_w_b, &conv_b_b, &dt_w, &bc_w, &dt_bias, &A_log, &D, &key_norm});
  py::gil_scoped_release release;
  return CoreFn::apply(zx, h0, dist, weights_, conv_w_f, conv_b_f, conv_w_b, conv_b_b, dt_w, bc_w, dt_bias, A_log, D, key_norm,
                       d_inner, nheads, ngroups, lo, hi, key_eps);
}

// MultiHeadISSMScan.forward as a whole (dest_module.py:515-585) for the configuration CoreFn is built for.
std::vector<Tensor> scan_layer(const Tensor& in_key, const Tensor& in_query, const Tensor& dist, const MaybeTensor& weights_,
                               const Tensor& key_proj, const Tensor& query_proj, const Tensor& out_key_proj,
                               const Tensor& out_query_proj, const Tensor& conv_w_f, const Tensor& conv_b_f, const Tensor& conv_w_b,
                               const Tensor& conv_b_b, const Tensor& dt_w, const Tensor& bc_w, const Tensor& dt_bias,
                               const Tensor& A_log, const Tensor& D, const Tensor& key_norm, double key_eps,
                               const MaybeTensor& query_w, const MaybeTensor& query_b, double query_eps,
                               int64_t d_inner, int64_t nheads, int64_t ngroups, double lo, double hi) {
  check_core(in_key, in_query, dist, opt(weights_), d_inner, nheads, ngroups,
             {&conv_w_f, &conv_b_f, &conv_w_b, &conv_b_b, &dt_w, &bc_w, &dt_bias, &A_log, &D, &key_norm});
  py::gil_scoped_release release;
  // Nothing to differentiate, bf16 and not too many tokens (chain_products): six or seven launches a layer where the separate steps take fifteen, and
  // no autograd nodes (six layers, 1024 tokens, 256 queries: 871 us -> 571 with eight launches; 524 -> 474 with six for eight behind faster
  // kernels; 3, 4 and 8 such scenes, which took the separate steps, 1047 -> 869, 1209 -> 1034 and 1990 -> 1788).
  const Tensor query_wt = opt(query_w), query_bt = opt(query_b), wts = opt(weights_);
  auto plain_bf16 = [&](const Tensor& t) {
    return !t.defined() || (t.scalar_type() == at::kBFloat16 && t.is_contiguous() && t.device() == in_key.device() &&
                            t.dim() == 1 && t.size(0) == d_inner && own_memory(t));
  };
  const double most = chain_products(d_inner);
  // (functorch's transforms refuse autograd functions, and so this path too)
  bool plain = !at::autocast::is_autocast_enabled(at::kCUDA) &&
               !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && few_tokens(in_key, key_proj, most) &&
               few_tokens(in_query, query_proj, most) && few_tokens(in_key, out_key_proj, most) &&
               few_tokens(in_query, out_query_proj, most) && in_query.device() == in_key.device() &&
               in_key.size(-1) == d_inner && in_query.size(-1) == d_inner && query_proj.size(0) == d_inner && d_inner % 4 == 0 &&
               d_inner <= 1024 && plain_bf16(key_norm) && plain_bf16(query_wt) && plain_bf16(query_bt);
  for (const Tensor* t : std::initializer_list<const Tensor*>{&in_key, &in_query, &dist, &key_proj, &query_proj, &out_key_proj,
                                                              &out_query_proj, &conv_w_f, &conv_w_b, &conv_b_f, &conv_b_b, &dt_w,
                                                              &bc_w, &dt_bias, &A_log, &D, &key_norm, &query_wt, &query_bt, &wts}) {
    if (!plain) break;
    plain = !t->defined() || (own_memory(*t) && !(at::GradMode::is_enabled() && t->requires_grad()) && !t->_fw_grad(0).defined());
  }
  // A run that another is to repeat takes the kernels of one with gradients.
  plain = plain && !runs_twice() && !(in_key.requires_grad() || in_query.requires_grad() || dist.requires_grad());
  if (plain) {
    const c10::DeviceGuard guard(in_key.device());
    const int64_t B = in_key.size(0), Ln = in_key.size(1), H = nheads, G = ngroups, di = d_inner, P = di / H, Cc = di + 2 * G,
                  K = dist.size(2), W = key_proj.size(0);
    CoreFn::check_sizes(W, conv_w_f, conv_w_b, conv_b_f, conv_b_b, dt_w, bc_w, dt_bias, A_log, D, key_norm, di, H, G);
    void* const stream = stream_of(in_key);
    issm_scan_args s{};
    s.dims = issm_dims{(int32_t)B, (int32_t)Ln, (int32_t)H, (int32_t)P, (int32_t)K, (int32_t)G, ISSM_CHUNK, 2};
    s.io_dtype = s.dt_dtype = s.h0_dtype = ISSM_BF16;
    size_t ws_bytes = 0;
    check(issm_fwd_workspace_bytes(&s, &ws_bytes), "workspace query");
    // one allocation for all that lies between the inputs and the outputs (seventeen were 24 us of host time)
    int64_t off[CoreFn::NSMALL + 1];
    const std::array<const Tensor*, CoreFn::NSMALL> arrays{&conv_w_f, &conv_w_b, &conv_b_f, &conv_b_b, &dt_w, &bc_w, &dt_bias,
                                                           &A_log, &D};
    const int64_t nflat = CoreFn::offsets(arrays, off);
    const Tensor d = cast(dist, at::kBFloat16).contiguous(), wt = f32c(wts);
    const bool joined = B * Ln * (K % 2 ? K : K / 2) <= JOINED_THREADS;
    enum { ZX, H0, FLAT, A1, X, TAIL, PRE, DT, BC, Y, LAST, WS, PARTS };
    const int64_t bytes[PARTS] = {2 * B * Ln * W, 2 * B * di * K, 4 * nflat, 4 * H * K, 4 * B * Ln * di, joined ? 0 : 8 * B * Ln * G,
                                  joined ? 0 : 4 * B * Ln * Cc, 2 * B * Ln * H * K, 8 * B * Ln * G * K, 4 * B * Ln * di, 8 * B * di * K,
                                  (int64_t)ws_bytes};
    int64_t at_[PARTS + 1] = {0};
    for (int i = 0; i < PARTS; ++i) at_[i + 1] = at_[i] + (bytes[i] + 255) / 256 * 256;
    const Tensor arena = fresh({at_[PARTS]}, in_key, at::kByte);
    char* const base = data<char>(arena);
    auto part = [&](int i, int64_t byte = 0) -> void* { return base + at_[i] + byte; };
    float *const par = (float*)part(FLAT), *const last = (float*)part(LAST);
    // the projections, the queries' into the layout of the scan's states
    auto product = [&](const Tensor& x, const void* px, const Tensor& w, void* y, int64_t turn) {
      return issm_linear_job{px, data(w), y, x.numel() / x.size(-1), (int32_t)w.size(1), (int32_t)w.size(0), (int32_t)turn};
    };
    issm_linear_args lin{};
    lin.njobs = 2;
    lin.dtype = ISSM_BF16;
    lin.stream = stream;
    lin.job[0] = product(in_key, data(in_key), key_proj, part(ZX), 0);
    lin.job[1] = product(in_query, data(in_query), query_proj, part(H0), K);
    CoreFn::small_parameters(arrays, K, par, (float*)part(A1), stream, &lin);
    void* bc[4];
    for (int i = 0; i < 4; ++i) bc[i] = part(BC, i * 2 * B * Ln * G * K);
    {
      issm_dwconv_args c{};
      c.batch = (int32_t)B;
      c.seqlen = (int32_t)Ln;
      c.channels = (int32_t)Cc;
      c.nsets = 2;
      c.taps = TAPS;
      c.dtype = ISSM_BF16;
      c.u = part(ZX, 2 * di);
      c.u_batch_stride = Ln * W;
      c.u_token_stride = W;
      c.chain = 1;
      c.stream = stream;
      c.w = par;
      c.bias = par + off[CoreFn::CB_F];
      c.y = part(X);
      c.split = (int32_t)di;
      issm_pgen_args a = pgen_args(d, par + off[CoreFn::DT_W], H, G);
      a.tok = part(ZX, 2 * (di + Cc));
      a.tok_stride = W;
      a.tok_add = par + off[CoreFn::DT_BIAS];
      a.dt = part(DT);
      a.Bm = bc[0];
      a.Cm = bc[1];
      a.Bm_back = bc[2];
      a.Cm_back = bc[3];
      a.weights = data<const float>(wt);
      if (joined) {
        check(issm_conv_param_gen_fwd(&c, &a), "issm_conv_param_gen_fwd");
      } else {
        c.pre = part(PRE);
        a.tail = c.y_tail = part(TAIL);
        check(issm_dwconv_silu_fwd(&c), "issm_dwconv_silu_fwd");
        check(issm_param_gen_fwd_only(&a), "issm_param_gen_fwd_only");
      }
    }
    s.flags = (wt.defined() ? 0u : ISSM_FLAG_DT_SOFTPLUS) | (D.dim() == 2 ? ISSM_FLAG_D_HAS_HDIM : 0u);
    s.dt_min = (float)lo;
    s.dt_max = (float)std::min(hi, 3.0e38);
    for (int i = 0; i < 2; ++i) {
      s.x[i] = issm_tensor{part(X, i * 2 * B * Ln * di), {Ln * di, di, P}};
      s.Bm[i] = issm_tensor{bc[2 * i], {Ln * G * K, G * K, K}};
      s.Cm[i] = issm_tensor{bc[2 * i + 1], {Ln * G * K, G * K, K}};
      s.out[i] = issm_tensor{part(Y, i * 2 * B * Ln * di), {Ln * di, di, P}};
      s.final_states[i] = last + i * B * di * K;
    }
    s.dt = issm_tensor{part(DT), {Ln * H * K, H * K, K}};
    s.h0 = issm_tensor{part(H0), {di * K, P * K, K}};
    s.A = (const float*)part(A1);
    s.D = par + off[CoreFn::D_];
    s.workspace = part(WS);
    s.workspace_bytes = ws_bytes;
    s.stream = stream;
    check(issm_scan_fwd_only(&s), "issm_scan_fwd_only");
    const Tensor out_key = fresh({B, Ln, out_key_proj.size(0)}, in_key, at::kBFloat16),
                 out_query = fresh({B, K, out_query_proj.size(0)}, in_key, at::kBFloat16);
    lin.job[0] = product(in_key, nullptr, out_key_proj, data(out_key), 0);
    lin.job[1] = product(in_query, nullptr, out_query_proj, data(out_query), 0);
    {
      issm_layer_out_args a{};
      a.batch = (int32_t)B;
      a.seqlen = (int32_t)Ln;
      a.queries = (int32_t)K;
      a.d_inner = (int32_t)di;
      a.dtype = ISSM_BF16;
      for (int i = 0; i < 2; ++i) {
        a.y[i] = s.out[i].ptr;
        a.last[i] = s.final_states[i];
      }
      a.z = part(ZX);
      a.z_row_stride = W;
      a.key_weight = data(key_norm);
      a.key_eps = (float)(4.0 * key_eps);
      a.query_weight = data(query_wt);
      a.query_bias = data(query_bt);
      a.query_eps = (float)query_eps;
      a.stream = stream;
      check(issm_layer_end(&a, &lin), "issm_layer_end");
    }
    return {out_key, out_query};
  }
  const variable_list in = linear_pair(in_key, key_proj, in_query, query_proj);
  variable_list core = CoreFn::apply(in[0], in[1], dist, weights_, conv_w_f, conv_b_f, conv_w_b, conv_b_b, dt_w, bc_w, dt_bias, A_log, D,
                                     key_norm, d_inner, nheads, ngroups, lo, hi, key_eps);
  const Tensor q = at::layer_norm(core[1], {d_inner}, query_w, query_b, query_eps);
  return linear_pair(core[0], out_key_proj, q, out_query_proj);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("scan", &scan);
  m.def("biscan", &biscan);
  m.def("scan_args", &scan_args);
  m.def("norm", &norm);
  m.def("norm_args", [](const Tensor& x, const MaybeTensor& z, const Tensor& w, const MaybeTensor& bias, double eps, int64_t group,
                        bool before_gate, bool layer_norm) {
    const issm_norm_args a = norm_args(x, opt(z), w, opt(bias), eps, group, before_gate, layer_norm);
    return py::bytes((const char*)&a, sizeof a);
  });
  m.def("linear_tokens", [](const Tensor& x, const Tensor& w) {
    py::gil_scoped_release release;
    return linear_tokens(x, w);
  });
  m.def("linear_pair", [](const Tensor& x0, const Tensor& w0, const Tensor& x1, const Tensor& w1) {
    py::gil_scoped_release release;
    return linear_pair(x0, w0, x1, w1);
  });
  m.def("runs_twice", &runs_twice);
  m.def("scan_core", &scan_core);
  m.def("scan_layer", &scan_layer);
}
