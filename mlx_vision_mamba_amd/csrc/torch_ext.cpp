// The host path of the package in C++: the autograd Functions of the scan,
// the conv, the LayerNorm and the Mamba block core, and the raw launches they
// share, over the C ABI of libmvm_scan.so (include/mvm_*.h).
//
// Why here and not in Python: a pass of the small workloads is a handful of
// launches of 5-20 us each, and the Python autograd Functions with their
// ctypes calls took 2-6 times as long to issue them as the GPU to run them
// (scan at B=2 L=196 D=1536, forward + VJP: 49 us of kernels in a pass of
// 252 us; LayerNorm of 6272 rows: 24 us in 150 us).  The functions below do
// what the Python ones did, in the same order: same checks, dtypes, layouts,
// saved tensors and gradients.
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <atomic>
#include <initializer_list>
#include <string>
#include <vector>

#include "mvm_conv.h"
#include "mvm_gemm.h"
#include "mvm_norm.h"
#include "mvm_scan.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// ----------------------------------------------------------------- errors

// a negative status of the library; becomes _lib.ScanError in Python
struct StatusError : std::runtime_error {
  int64_t code;
  explicit StatusError(int64_t c)
      : std::runtime_error("libmvm_scan error " + std::to_string(c) + ": " + mvm_last_error()), code(c) {}
};

int64_t check(int64_t rc) {
  if (rc < 0) throw StatusError(rc);
  return rc;
}

[[noreturn]] void bad_value(const std::string& msg) { throw py::value_error(msg); }

std::string shape_str(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

// sets the Python error that stands for e (with the GIL held)
void set_scan_error(const StatusError& e) {
  const std::string msg = e.what();
  const py::object cls = py::module_::import("mlx_vision_mamba_amd._lib").attr("ScanError");
  const auto cut = msg.find(": ");
  const py::object exc = cls(e.code, msg.substr(cut == std::string::npos ? 0 : cut + 2));
  PyErr_SetObject(cls.ptr(), exc.ptr());
}

// Runs f with torch's exception translation, and StatusError as ScanError
template <typename F>
auto guarded(F&& f) -> decltype(f()) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const StatusError& e) {
    set_scan_error(e);
    throw py::error_already_set();
  }
  END_HANDLE_TH_ERRORS_PYBIND
}

// Runs a Function's backward: the autograd engine carries its exceptions from
// its own threads to the caller's, but hands a C++ one over as RuntimeError.
// Library refusals and ValueErrors travel as the Python exceptions they are.
template <typename F>
variable_list in_backward(F&& f) {
  python_error err;
  try {
    return f();
  } catch (const StatusError& e) {
    py::gil_scoped_acquire gil;
    set_scan_error(e);
    err.persist();
  } catch (const py::builtin_exception& e) {
    py::gil_scoped_acquire gil;
    e.set_error();
    err.persist();
  }
  throw python_error(std::move(err));
}

// ---------------------------------------------------------------- helpers

const float* fp(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.const_data_ptr()) : nullptr; }
float* fpm(const Tensor& t) { return t.defined() ? static_cast<float*>(t.mutable_data_ptr()) : nullptr; }

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

Tensor empty_like_opts(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dt = at::kFloat) {
  return at::empty(sizes, like.options().dtype(dt).requires_grad(false));
}

Tensor workspace(int64_t nbytes, const Tensor& like) {
  return empty_like_opts({std::max<int64_t>(nbytes, 1)}, like, at::kByte);
}

void check_device(std::initializer_list<const Tensor*> ts) {
  const auto dev = (*ts.begin())->device();
  TORCH_CHECK(dev.is_cuda(), "mlx_vision_mamba_amd scans run only on the GPU (HIP); got tensors on ", dev,
              ". There is no CPU fallback.");
  for (const Tensor* t : ts)
    TORCH_CHECK(!t->defined() || t->device() == dev, "all scan tensors must be on ", dev, "; got one on ",
                t->device());
}

// true when no two elements of t share memory: ordered by stride, each
// dimension's stride clears the span of the smaller ones
bool no_overlap(const Tensor& t) {
  std::vector<std::pair<int64_t, int64_t>> v;
  for (int64_t i = 0; i < t.dim(); ++i)
    if (t.size(i) != 1) v.emplace_back(t.stride(i), t.size(i));
  std::sort(v.begin(), v.end());
  int64_t span = 1;
  for (const auto& p : v) {
    if (p.first < span) return false;
    span = p.first * p.second;
  }
  return true;
}

bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) == 0; }

// The gradients `out` of a Function whose backward is raw launches, as they
// leave it.  Under create_graph they would have no history, and a derivative
// through them would silently lack this Function's part: they get a node that
// raises instead, on the paths to the Function's inputs and to the incoming
// gradients.  (The gradients themselves are right and may be used.)
variable_list once_differentiable(variable_list out, const variable_list& grads, const char* what) {
  if (!at::GradMode::is_enabled()) return out;
  auto edges = torch::autograd::collect_next_edges(grads);
  if (const auto node = torch::autograd::get_current_node())
    for (const auto& e : node->next_edges())
      if (e.is_valid()) edges.push_back(e);
  const auto err = std::make_shared<torch::autograd::Error>(std::string(what) + " is not twice differentiable",
                                                            std::move(edges));
  for (Tensor& t : out)
    if (t.defined()) {
      t = t.detach();
      torch::autograd::create_gradient_edge(t, err);
    }
  return out;
}

// -------------------------------------------------------- launch timing
//
// scan.set_scan_timing's records: the Python callables that open and close
// one record, called around each scan launch while timing is on.
std::atomic<bool> g_timing{false};
py::object* g_timer_start = nullptr;
py::object* g_timer_stop = nullptr;

class Timed {
 public:
  explicit Timed(const char* kind) : kind_(kind) {
    if (!g_timing.load()) return;
    py::gil_scoped_acquire gil;
    rec_ = new py::object((*g_timer_start)());
  }
  ~Timed() {
    if (rec_ == nullptr) return;
    py::gil_scoped_acquire gil;
    delete rec_;
  }
  void stop(int64_t fwd_bytes, int64_t vjp_bytes) {
    if (rec_ == nullptr) return;
    py::gil_scoped_acquire gil;
    (*g_timer_stop)(*rec_, kind_, kind_[0] == 'f' ? fwd_bytes : vjp_bytes);
  }

 private:
  const char* kind_;
  py::object* rec_ = nullptr;
};

// bytes of a scan forward / VJP, every tensor once (scan.algorithmic_bytes)
std::pair<int64_t, int64_t> scan_bytes(int64_t rows, int64_t L, int64_t D, int64_t N, int64_t in, int64_t out,
                                       int64_t K) {
  return {rows * L * D * (in + 4 + out) + rows * L * N * 2 * in + K * (D * N * 4 + D * 4),
          rows * L * D * (in + 4 + in + out + 4) + rows * L * N * (2 * in + 2 * out) + K * (D * N * 8 + D * 8)};
}
std::pair<int64_t, int64_t> fused_bytes(int64_t rows, int64_t L, int64_t D, int64_t N, int64_t K, bool gate,
                                        bool bias) {
  auto b = scan_bytes(rows, L, D, N, 4, 4, K);
  if (gate) {
    b.first += rows * L * D * 8;
    b.second += rows * L * D * 12;
  }
  if (bias) {
    b.first += K * D * 4;
    b.second += K * D * 8;
  }
  return b;
}

// -------------------------------------------------------------- plain scan

mvm_scan_desc make_desc(const Tensor& u, const Tensor& Bm, at::ScalarType in_dt, at::ScalarType out_dt,
                        const Tensor& tok, int64_t chunk_len) {
  mvm_scan_desc d{};
  d.batch = u.size(0); d.seqlen = u.size(1); d.ndir = u.size(2); d.dim = u.size(3);
  d.dstate = Bm.size(3);
  d.x_stride_b = u.stride(0); d.x_stride_t = u.stride(1); d.x_stride_k = u.stride(2);
  d.bc_stride_b = Bm.stride(0); d.bc_stride_t = Bm.stride(1); d.bc_stride_k = Bm.stride(2);
  d.seq_to_tok = tok.defined() ? static_cast<const int32_t*>(tok.const_data_ptr()) : nullptr;
  d.in_dtype = in_dt == at::kBFloat16 ? MVM_BF16 : MVM_F32;
  d.out_dtype = out_dt == at::kBFloat16 ? MVM_BF16 : MVM_F32;
  d.chunk_len = static_cast<int32_t>(chunk_len);
  return d;
}

struct ScanIn {
  Tensor u, delta, A, Bm, Cm, Dv;
  at::ScalarType in_dt;
};

// canonical dtypes and layouts; shapes are (B,L,K,D), (K,D,N), (B,L,K,N), (K,D)
ScanIn prepare(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& Bm, const Tensor& Cm,
               const Tensor& Dv) {
  if (u.dim() != 4 || delta.sizes() != u.sizes())
    bad_value("u and delta must be (B, L, K, D) of equal shape; got " + shape_str(u) + ", " + shape_str(delta));
  const int64_t bsz = u.size(0), L = u.size(1), K = u.size(2), D = u.size(3);
  if (A.dim() != 3 || A.size(0) != K || A.size(1) != D)
    bad_value("A must be (K=" + std::to_string(K) + ", D=" + std::to_string(D) + ", N); got " + shape_str(A));
  const int64_t N = A.size(2);
  if (N < 1 || N > MVM_MAX_DSTATE)
    bad_value("d_state=" + std::to_string(N) + " unsupported (1.." + std::to_string(MVM_MAX_DSTATE) + ")");
  const std::vector<int64_t> bc = {bsz, L, K, N};
  if (Bm.sizes() != bc || Cm.sizes() != bc)
    bad_value("B and C must be (" + std::to_string(bsz) + ", " + std::to_string(L) + ", " + std::to_string(K) +
              ", " + std::to_string(N) + "); got " + shape_str(Bm) + ", " + shape_str(Cm));
  if (Dv.dim() != 2 || Dv.size(0) != K || Dv.size(1) != D)
    bad_value("D must be (" + std::to_string(K) + ", " + std::to_string(D) + "); got " + shape_str(Dv));
  check_device({&u, &delta, &A, &Bm, &Cm, &Dv});
  ScanIn s;
  const bool bf = u.scalar_type() == at::kBFloat16 && Bm.scalar_type() == at::kBFloat16 &&
                  Cm.scalar_type() == at::kBFloat16;
  s.in_dt = bf ? at::kBFloat16 : at::kFloat;
  s.u = u.to(s.in_dt).contiguous();
  s.Bm = Bm.to(s.in_dt);
  s.Cm = Cm.to(s.in_dt);
  // views (e.g. column slices of a projection output) are kept when they
  // share strides and no two elements overlap
  bool keep = s.Bm.strides() == s.Cm.strides() && s.Bm.stride(3) == 1 && no_overlap(s.Bm);
  for (int64_t st : s.Bm.strides()) keep = keep && st >= 0;
  if (!keep) {
    s.Bm = s.Bm.contiguous();
    s.Cm = s.Cm.contiguous();
  }
  s.delta = delta.to(at::kFloat).contiguous();
  s.A = A.to(at::kFloat).contiguous();
  s.Dv = Dv.to(at::kFloat).contiguous();
  return s;
}

at::ScalarType out_type(std::optional<at::ScalarType> dt, at::ScalarType in_dt) {
  const at::ScalarType t = dt.value_or(in_dt);
  if (t != at::kFloat && t != at::kBFloat16)
    throw py::key_error(std::string("unsupported out_dtype ") + c10::toString(t));
  return t;
}

// (y, checkpoints); y is (B, L, D) when flat.  It is allocated in that shape:
// a view made inside a Function could not be changed in place
std::pair<Tensor, Tensor> scan_fwd(const ScanIn& s, const Tensor& tok, int64_t chunk_len,
                                   std::optional<at::ScalarType> out_dtype, bool save_ckpt, bool flat) {
  const auto out_dt = out_type(out_dtype, s.in_dt);
  const auto d = make_desc(s.u, s.Bm, s.in_dt, out_dt, tok, chunk_len);
  c10::OptionalDeviceGuard guard(s.u.device());
  Tensor y = flat ? empty_like_opts({s.u.size(0), s.u.size(1), s.u.size(3)}, s.u, out_dt)
                  : empty_like_opts(s.u.sizes(), s.u, out_dt);
  Tensor ckpt;
  if (save_ckpt) ckpt = empty_like_opts({check(mvm_scan_ckpt_elems(&d))}, s.u);
  const int64_t nbytes = check(mvm_scan_workspace_bytes(&d, 0));
  const Tensor ws = workspace(nbytes, s.u);
  Timed timed("fwd");
  check(mvm_scan_fwd(&d, s.u.const_data_ptr(), fp(s.delta), fp(s.A), s.Bm.const_data_ptr(),
                     s.Cm.const_data_ptr(), fp(s.Dv), y.mutable_data_ptr(), fpm(ckpt),
                     ws.mutable_data_ptr(), static_cast<size_t>(nbytes), stream_of(s.u)));
  const auto nb = scan_bytes(d.batch * d.ndir, d.seqlen, d.dim, d.dstate, c10::elementSize(s.in_dt),
                             c10::elementSize(out_dt), d.ndir);
  timed.stop(nb.first, nb.second);
  return {y, ckpt};
}

std::vector<Tensor> scan_bwd(const ScanIn& s, Tensor dy, const Tensor& ckpt, const Tensor& tok, int64_t chunk_len,
                             std::optional<at::ScalarType> out_dtype) {
  const auto out_dt = out_type(out_dtype, s.in_dt);
  const auto d = make_desc(s.u, s.Bm, s.in_dt, out_dt, tok, chunk_len);
  dy = dy.to(s.in_dt).contiguous();
  if (dy.sizes() != s.u.sizes()) bad_value("dy shape " + shape_str(dy) + " != " + shape_str(s.u));
  c10::OptionalDeviceGuard guard(s.u.device());
  const auto opt = s.u.options().requires_grad(false);
  Tensor du = at::empty(s.u.sizes(), opt.dtype(out_dt));
  Tensor ddelta = at::empty(s.u.sizes(), opt.dtype(at::kFloat));
  Tensor dA = at::empty(s.A.sizes(), opt.dtype(at::kFloat));
  Tensor dB = at::empty_strided(s.Bm.sizes(), s.Bm.strides(), opt.dtype(out_dt));
  Tensor dC = at::empty_strided(s.Bm.sizes(), s.Bm.strides(), opt.dtype(out_dt));
  Tensor dD = at::empty(s.Dv.sizes(), opt.dtype(at::kFloat));
  const int64_t nbytes = check(mvm_scan_workspace_bytes(&d, ckpt.defined() ? 1 : 2));
  const Tensor ws = workspace(nbytes, s.u);
  Timed timed("bwd");
  check(mvm_scan_bwd(&d, s.u.const_data_ptr(), fp(s.delta), fp(s.A), s.Bm.const_data_ptr(),
                     s.Cm.const_data_ptr(), fp(s.Dv), fp(ckpt), dy.const_data_ptr(), du.mutable_data_ptr(),
                     fpm(ddelta), fpm(dA), dB.mutable_data_ptr(), dC.mutable_data_ptr(), fpm(dD),
                     ws.mutable_data_ptr(), static_cast<size_t>(nbytes), stream_of(s.u)));
  const auto nb = scan_bytes(d.batch * d.ndir, d.seqlen, d.dim, d.dstate, c10::elementSize(s.in_dt),
                             c10::elementSize(out_dt), d.ndir);
  timed.stop(nb.first, nb.second);
  return {du, ddelta, dA, dB, dC, dD};
}

// the (B, L, D) form: one direction, inserted as dimension 2 (0 for A and D)
std::vector<Tensor> lift(const std::vector<Tensor>& t, bool flat) {
  if (!flat) return t;
  return {t[0].unsqueeze(2), t[1].unsqueeze(2), t[2].unsqueeze(0),
          t[3].unsqueeze(2), t[4].unsqueeze(2), t[5].unsqueeze(0)};
}

// y = scan(u, delta, A, B, C, D) with the fused HIP VJP (the
// custom_function + vjp pair of mamba_metal_fused.py:229-250)
struct ScanFn : Function<ScanFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& u, const Tensor& delta, const Tensor& A,
                        const Tensor& Bm, const Tensor& Cm, const Tensor& Dv, const OptTensor& tok_,
                        int64_t chunk_len, std::optional<at::ScalarType> out_dtype, bool needs, bool flat) {
    const Tensor tok = tok_.value_or(Tensor());
    const auto t = lift({u, delta, A, Bm, Cm, Dv}, flat);
    auto [y, ckpt] = scan_fwd(prepare(t[0], t[1], t[2], t[3], t[4], t[5]), tok, chunk_len, out_dtype, needs,
                              flat);
    ctx->saved_data["chunk"] = chunk_len;
    ctx->saved_data["out"] = out_dtype.has_value() ? static_cast<int64_t>(*out_dtype) : int64_t{-1};
    ctx->saved_data["flat"] = flat;
    if (needs) ctx->save_for_backward({u, delta, A, Bm, Cm, Dv, ckpt, tok});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return grads(ctx, g); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& g) {
    const auto sv = ctx->get_saved_variables();
    const bool flat = ctx->saved_data["flat"].toBool();
    const int64_t od = ctx->saved_data["out"].toInt();
    variable_list out;
    {
      at::NoGradGuard no_grad;
      const auto t = lift({sv[0], sv[1], sv[2], sv[3], sv[4], sv[5]}, flat);
      out = scan_bwd(prepare(t[0], t[1], t[2], t[3], t[4], t[5]), flat ? g[0].unsqueeze(2) : g[0], sv[6], sv[7],
                     ctx->saved_data["chunk"].toInt(),
                     od < 0 ? std::nullopt : std::make_optional(static_cast<at::ScalarType>(od)));
      for (int i = 0; i < 6; ++i) {
        out[i] = out[i].to(sv[i].scalar_type());
        if (flat) out[i] = out[i].squeeze(i == 2 || i == 5 ? 0 : 2);
      }
    }
    out.resize(11);
    return once_differentiable(std::move(out), g, "the selective scan");
  }
};

Tensor scan(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& Bm, const Tensor& Cm,
            const Tensor& Dv, const OptTensor& tok, int64_t chunk_len, std::optional<at::ScalarType> out_dtype,
            bool flat) {
  return guarded([&] {
    // checkpoints only when a gradient can be asked for
    bool needs = false;
    for (const Tensor* t : {&u, &delta, &A, &Bm, &Cm, &Dv}) needs = needs || t->requires_grad();
    return ScanFn::apply(u, delta, A, Bm, Cm, Dv, tok, chunk_len, out_dtype,
                         needs && at::GradMode::is_enabled(), flat);
  });
}

std::pair<Tensor, OptTensor> scan_forward(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& Bm,
                                          const Tensor& Cm, const Tensor& Dv, const OptTensor& tok,
                                          int64_t chunk_len, std::optional<at::ScalarType> out_dtype,
                                          bool save_ckpt, bool flat) {
  return guarded([&]() -> std::pair<Tensor, OptTensor> {
    const auto t = lift({u, delta, A, Bm, Cm, Dv}, flat);
    auto [y, ckpt] = scan_fwd(prepare(t[0], t[1], t[2], t[3], t[4], t[5]), tok.value_or(Tensor()), chunk_len,
                              out_dtype, save_ckpt, flat);
    return {y, ckpt.defined() ? OptTensor(ckpt) : std::nullopt};
  });
}

std::vector<Tensor> scan_backward(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& Bm,
                                  const Tensor& Cm, const Tensor& Dv, const Tensor& dy, const OptTensor& ckpt,
                                  const OptTensor& tok, int64_t chunk_len,
                                  std::optional<at::ScalarType> out_dtype) {
  return guarded([&] {
    return scan_bwd(prepare(u, delta, A, Bm, Cm, Dv), dy, ckpt.value_or(Tensor()), tok.value_or(Tensor()),
                    chunk_len, out_dtype);
  });
}

// -------------------------------------------------------------- fused scan

mvm_scan_fused_desc fused_desc(const Tensor& u, const Tensor& delta_raw, const Tensor& Bm, const Tensor& y,
                               const Tensor& z, const Tensor& tok, int64_t chunk_len, bool a_is_log) {
  mvm_scan_fused_desc f{};
  f.scan = make_desc(u, Bm, at::kFloat, at::kFloat, tok, chunk_len);
  f.a_is_log = a_is_log;
  f.dt_stride_b = delta_raw.stride(0); f.dt_stride_t = delta_raw.stride(1); f.dt_stride_k = delta_raw.stride(2);
  f.y_stride_b = y.stride(0); f.y_stride_t = y.stride(1); f.y_stride_k = y.stride(2);
  if (z.defined()) {
    f.z_stride_b = z.stride(0); f.z_stride_t = z.stride(1); f.z_stride_k = z.stride(2);
  }
  return f;
}

void check_fused(const Tensor& u, const Tensor& delta_raw, const Tensor& dbias, const Tensor& A, const Tensor& Bm,
                 const Tensor& Cm, const Tensor& Dv, const Tensor& z) {
  if (u.dim() != 4 || A.dim() < 1) bad_value("u must be (B, L, K, D)");
  const int64_t bsz = u.size(0), L = u.size(1), K = u.size(2), D = u.size(3), N = A.size(-1);
  if (delta_raw.sizes() != u.sizes() || (z.defined() && z.sizes() != u.sizes()))
    bad_value("u, delta_raw and z must share the (B, L, K, D) shape");
  if (A.sizes() != at::IntArrayRef({K, D, N}) || Bm.sizes() != at::IntArrayRef({bsz, L, K, N}) ||
      Cm.sizes() != Bm.sizes())
    bad_value("A must be (K, D, N) and B, C (B, L, K, N)");
  if (Dv.sizes() != at::IntArrayRef({K, D}) || (dbias.defined() && dbias.sizes() != at::IntArrayRef({K, D})))
    bad_value("D and the dt bias must be (K, D)");
  if (Bm.strides() != Cm.strides()) bad_value("B and C must share strides");
  check_device({&u, &delta_raw, &A, &Bm, &Cm, &Dv, &dbias, &z});
  for (const Tensor* t : {&u, &delta_raw, &A, &Bm, &Cm, &Dv, &dbias, &z})
    if (t->defined() && (t->scalar_type() != at::kFloat || t->stride(-1) != 1))
      bad_value("the fused scan takes float32 views with channel stride 1");
  if (!A.is_contiguous() || !Dv.is_contiguous() || (dbias.defined() && !dbias.is_contiguous()))
    bad_value("A, D and the dt bias must be contiguous");
}

struct FusedOut {
  Tensor y, y_raw, ckpt;
};
// delta_raw is read; or, with dt (B, L, K, R) in rows of B's strides and W_dt
// (K, D, R), formed in the kernel and written to delta_raw when saving
FusedOut fused_fwd(const Tensor& u, const Tensor& delta_raw, const Tensor& dbias, const Tensor& A,
                   const Tensor& Bm, const Tensor& Cm, const Tensor& Dv, const Tensor& z, const Tensor& tok,
                   int64_t chunk_len, bool save, bool a_is_log, const Tensor& dt = Tensor(),
                   const Tensor& W_dt = Tensor()) {
  check_fused(u, delta_raw, dbias, A, Bm, Cm, Dv, z);
  FusedOut o;
  c10::OptionalDeviceGuard guard(u.device());
  o.y = empty_like_opts(u.sizes(), u);
  const auto f = fused_desc(u, delta_raw, Bm, o.y, z, tok, chunk_len, a_is_log);
  if (save && z.defined()) o.y_raw = empty_like_opts(u.sizes(), u);
  if (save) o.ckpt = empty_like_opts({check(mvm_scan_ckpt_elems(&f.scan))}, u);
  const int64_t nbytes = check(mvm_scan_fused_workspace_bytes(&f, 0, z.defined()));
  const Tensor ws = workspace(nbytes, u);
  Timed timed("fwd");
  if (dt.defined())
    check(mvm_scan_fused_dt_fwd(&f, fp(u), fp(dt), static_cast<int32_t>(dt.size(3)), fp(W_dt), fp(dbias), fp(A),
                                fp(Bm), fp(Cm), fp(Dv), fp(z), fpm(o.y), fpm(o.y_raw),
                                save ? fpm(delta_raw) : nullptr, fpm(o.ckpt), ws.mutable_data_ptr(),
                                static_cast<size_t>(nbytes), stream_of(u)));
  else
    check(mvm_scan_fused_fwd(&f, fp(u), fp(delta_raw), fp(dbias), fp(A), fp(Bm), fp(Cm), fp(Dv), fp(z), fpm(o.y),
                             fpm(o.y_raw), fpm(o.ckpt), ws.mutable_data_ptr(), static_cast<size_t>(nbytes),
                             stream_of(u)));
  const auto nb = fused_bytes(u.size(0) * u.size(2), u.size(1), u.size(3), A.size(-1), u.size(2), z.defined(),
                              dbias.defined());
  timed.stop(nb.first, nb.second);
  return o;
}

struct FusedGrads {
  Tensor du, ddelta_raw, ddbias, dA, dB, dC, dD, dz;
};
// fills the views of g that are defined, allocates the others with the
// layout of their primal
void fused_bwd(const Tensor& u, const Tensor& delta_raw, const Tensor& dbias, const Tensor& A, const Tensor& Bm,
               const Tensor& Cm, const Tensor& Dv, const Tensor& z, const Tensor& y_raw, const Tensor& ckpt,
               Tensor dy, const Tensor& tok, int64_t chunk_len, bool a_is_log, FusedGrads& g) {
  check_fused(u, delta_raw, dbias, A, Bm, Cm, Dv, z);
  if (dy.sizes() != u.sizes()) bad_value("dy shape " + shape_str(dy) + " != " + shape_str(u));
  if (z.defined() && y_raw.defined() && !y_raw.is_contiguous()) bad_value("y_raw must be contiguous");
  dy = dy.to(at::kFloat).contiguous();
  c10::OptionalDeviceGuard guard(u.device());
  auto like = [](const Tensor& t) {
    // same strides as the primal (a layout with gaps allocates its span)
    if (!no_overlap(t)) bad_value("a primal whose elements overlap (e.g. broadcast) needs an output view");
    return at::empty_strided(t.sizes(), t.strides(), t.options().dtype(at::kFloat).requires_grad(false));
  };
  if (!g.du.defined()) g.du = like(u);
  if (!g.ddelta_raw.defined()) g.ddelta_raw = like(delta_raw);
  if (!g.dB.defined() || !g.dC.defined()) {
    g.dB = like(Bm);
    g.dC = like(Bm);
  }
  if (g.dB.strides() != Bm.strides() || g.dC.strides() != Bm.strides())
    bad_value("dB and dC must have the strides of B");
  if (z.defined() && !g.dz.defined()) g.dz = like(z);
  for (const Tensor* t : {&g.du, &g.ddelta_raw, &g.dB, &g.dC, z.defined() ? &g.dz : &g.du})
    if (!no_overlap(*t)) bad_value("gradient views must not overlap themselves");
  if ((z.defined() && g.dz.strides() != z.strides()) || g.ddelta_raw.strides() != delta_raw.strides() ||
      g.du.strides() != u.strides())
    bad_value("gradient views must have the strides of their primals");
  if (dbias.defined()) g.ddbias = empty_like_opts(dbias.sizes(), dbias);
  g.dA = empty_like_opts(A.sizes(), A);
  g.dD = empty_like_opts(Dv.sizes(), Dv);
  const auto f = fused_desc(u, delta_raw, Bm, dy, z, tok, chunk_len, a_is_log);
  const int64_t nbytes = check(mvm_scan_fused_workspace_bytes(&f, 1, z.defined()));
  const Tensor ws = workspace(nbytes, u);
  Timed timed("bwd");
  check(mvm_scan_fused_bwd(&f, fp(u), fp(delta_raw), fp(dbias), fp(A), fp(Bm), fp(Cm), fp(Dv), fp(z), fp(y_raw),
                           fp(ckpt), fp(dy), fpm(g.du), fpm(g.ddelta_raw), fpm(g.ddbias), fpm(g.dA), fpm(g.dB),
                           fpm(g.dC), fpm(g.dD), z.defined() ? fpm(g.dz) : nullptr, ws.mutable_data_ptr(),
                           static_cast<size_t>(nbytes), stream_of(u)));
  const auto nb = fused_bytes(u.size(0) * u.size(2), u.size(1), u.size(3), A.size(-1), u.size(2), z.defined(),
                              dbias.defined());
  timed.stop(nb.first, nb.second);
}

OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

std::tuple<Tensor, OptTensor, OptTensor> scan_fused_forward(const Tensor& u, const Tensor& delta_raw,
                                                            const OptTensor& dbias, const Tensor& A,
                                                            const Tensor& Bm, const Tensor& Cm, const Tensor& Dv,
                                                            const OptTensor& z, const OptTensor& tok,
                                                            int64_t chunk_len, bool save, bool a_is_log) {
  return guarded([&]() -> std::tuple<Tensor, OptTensor, OptTensor> {
    at::NoGradGuard no_grad;
    const auto o = fused_fwd(u, delta_raw, dbias.value_or(Tensor()), A, Bm, Cm, Dv, z.value_or(Tensor()),
                             tok.value_or(Tensor()), chunk_len, save, a_is_log);
    return {o.y, opt(o.y_raw), opt(o.ckpt)};
  });
}

std::tuple<Tensor, Tensor, OptTensor, Tensor, Tensor, Tensor, Tensor, OptTensor> scan_fused_backward(
    const Tensor& u, const Tensor& delta_raw, const OptTensor& dbias, const Tensor& A, const Tensor& Bm,
    const Tensor& Cm, const Tensor& Dv, const OptTensor& z, const OptTensor& y_raw, const OptTensor& ckpt,
    const Tensor& dy, const OptTensor& tok, int64_t chunk_len, const OptTensor& du, const OptTensor& ddelta_raw,
    const OptTensor& dB, const OptTensor& dC, const OptTensor& dz, bool a_is_log) {
  return guarded([&]() -> std::tuple<Tensor, Tensor, OptTensor, Tensor, Tensor, Tensor, Tensor, OptTensor> {
    at::NoGradGuard no_grad;
    FusedGrads g;
    g.du = du.value_or(Tensor());
    g.ddelta_raw = ddelta_raw.value_or(Tensor());
    g.dB = dB.value_or(Tensor());
    g.dC = dC.value_or(Tensor());
    g.dz = dz.value_or(Tensor());
    fused_bwd(u, delta_raw, dbias.value_or(Tensor()), A, Bm, Cm, Dv, z.value_or(Tensor()),
              y_raw.value_or(Tensor()), ckpt.value_or(Tensor()), dy, tok.value_or(Tensor()), chunk_len, a_is_log, g);
    return {g.du, g.ddelta_raw, opt(g.ddbias), g.dA, g.dB, g.dC, g.dD, opt(g.dz)};
  });
}

// -------------------------------------------------------------------- conv

mvm_conv_desc conv_desc(const Tensor& x, const Tensor& y, const Tensor& dx, int64_t kc, const Tensor& tok) {
  mvm_conv_desc d{};
  d.batch = x.size(0); d.seqlen = x.size(1); d.ndir = x.size(2); d.dim = x.size(3);
  d.kwidth = kc;
  d.x_stride_b = x.stride(0); d.x_stride_t = x.stride(1); d.x_stride_k = x.stride(2);
  d.y_stride_b = y.stride(0); d.y_stride_t = y.stride(1); d.y_stride_k = y.stride(2);
  d.dx_stride_b = dx.stride(0); d.dx_stride_t = dx.stride(1); d.dx_stride_k = dx.stride(2);
  d.seq_to_tok = tok.defined() ? static_cast<const int32_t*>(tok.const_data_ptr()) : nullptr;
  return d;
}

// y (a (B, N, K, D) view with channel stride 1) = silu(conv(x) + b)
void conv_fwd(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& y, const Tensor& tok) {
  const auto d = conv_desc(x, y, y, w.size(2), tok);
  c10::OptionalDeviceGuard guard(x.device());
  check(mvm_conv_silu_fwd(&d, fp(x), fp(w), fp(b), fpm(y), stream_of(x)));
}

// writes dx (a view with its own strides); returns (dw, dbias)
std::pair<Tensor, Tensor> conv_bwd(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& dy,
                                   const Tensor& dx, const Tensor& tok) {
  Tensor dw = empty_like_opts(w.sizes(), w), db = empty_like_opts(b.sizes(), b);
  const auto d = conv_desc(x, dy, dx, w.size(2), tok);
  c10::OptionalDeviceGuard guard(x.device());
  const int64_t nbytes = check(mvm_conv_workspace_bytes(&d));
  const Tensor ws = workspace(nbytes, x);
  check(mvm_conv_silu_bwd(&d, fp(x), fp(w), fp(b), fp(dy), fpm(dx), fpm(dw), fpm(db), ws.mutable_data_ptr(),
                          static_cast<size_t>(nbytes), stream_of(x)));
  return {dw, db};
}

struct ConvFn : Function<ConvFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w_, const Tensor& b_,
                        const OptTensor& tok_) {
    check_device({&x_, &w_, &b_});
    const Tensor tok = tok_.value_or(Tensor());
    Tensor x = x_;
    if (x.dim() != 4 || x.stride(-1) != 1) x = x.contiguous();
    x = x.to(at::kFloat);
    const Tensor w = w_.to(at::kFloat).contiguous(), b = b_.to(at::kFloat).contiguous();
    Tensor y = empty_like_opts(x.sizes(), x);
    conv_fwd(x, w, b, y, tok);
    ctx->save_for_backward({x, w, b, tok});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return grads(ctx, g); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& g) {
    const auto sv = ctx->get_saved_variables();
    variable_list out;
    {
      at::NoGradGuard no_grad;
      Tensor dx = empty_like_opts(sv[0].sizes(), sv[0]);
      Tensor dy = g[0].to(at::kFloat).contiguous();
      // (one with no elements counts as contiguous whatever its strides)
      if (dy.strides() != dx.strides()) dy = dy.as_strided(dx.sizes(), dx.strides());
      auto [dw, db] = conv_bwd(sv[0], sv[1], sv[2], dy, dx, sv[3]);
      out = {dx, dw, db, Tensor()};
    }
    return once_differentiable(std::move(out), g, "the causal conv");
  }
};

Tensor conv_silu(const Tensor& x, const Tensor& w, const Tensor& b, const OptTensor& tok) {
  return guarded([&] { return ConvFn::apply(x, w, b, tok); });
}

// --------------------------------------------------------------- LayerNorm

struct NormFn : Function<NormFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Tensor& bias,
                               double eps, bool residual) {
    check_device({&x, &weight, &bias});
    const int64_t E = x.size(-1);
    if (weight.sizes() != at::IntArrayRef({E}) || bias.sizes() != at::IntArrayRef({E}))
      bad_value("weight and bias must be (" + std::to_string(E) + ",); got " + shape_str(weight) + ", " +
                shape_str(bias));
    const Tensor x2 = x.reshape({-1, E}).to(at::kFloat).contiguous();
    const Tensor w = weight.to(at::kFloat).contiguous(), b = bias.to(at::kFloat).contiguous();
    const int64_t R = x2.size(0);
    Tensor y = empty_like_opts({R, E}, x2), mean = empty_like_opts({R}, x2), rstd = empty_like_opts({R}, x2);
    const mvm_norm_desc d{R, E, E, E, static_cast<float>(eps), 0};
    c10::OptionalDeviceGuard guard(x.device());
    check(mvm_layernorm_fwd(&d, fp(x2), fp(w), fp(b), fpm(y), fpm(mean), fpm(rstd), stream_of(x)));
    ctx->save_for_backward({x2, w, mean, rstd});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->saved_data["types"] = std::vector<int64_t>{static_cast<int64_t>(x.scalar_type()),
                                                    static_cast<int64_t>(weight.scalar_type()),
                                                    static_cast<int64_t>(bias.scalar_type())};
    y = y.view(x.sizes()).to(x.scalar_type());
    if (residual) return {y, x};  // x itself: an alias whose gradient comes back here
    return {y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return once_differentiable(grads(ctx, g), g, "the LayerNorm"); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& g) {
    at::NoGradGuard no_grad;
    const auto sv = ctx->get_saved_variables();
    const Tensor &x2 = sv[0], &w = sv[1];
    const int64_t R = x2.size(0), E = x2.size(1);
    const Tensor dy = g[0].reshape({R, E}).to(at::kFloat).contiguous();
    Tensor dres;
    if (g.size() > 1 && g[1].defined()) dres = g[1].reshape({R, E}).to(at::kFloat).contiguous();
    Tensor dx = empty_like_opts({R, E}, x2), dw = empty_like_opts({E}, x2), db = empty_like_opts({E}, x2);
    const mvm_norm_desc d{R, E, E, E, static_cast<float>(ctx->saved_data["eps"].toDouble()), 0};
    c10::OptionalDeviceGuard guard(x2.device());
    const int64_t nbytes = check(mvm_norm_workspace_bytes(&d));
    const Tensor ws = workspace(nbytes, x2);
    check(mvm_layernorm_bwd(&d, fp(x2), fp(w), fp(sv[2]), fp(sv[3]), fp(dy), fp(dres), fpm(dx), fpm(dw), fpm(db),
                            ws.mutable_data_ptr(), static_cast<size_t>(nbytes), stream_of(x2)));
    const auto ty = ctx->saved_data["types"].toIntVector();
    const auto dt = [&](int i) { return static_cast<at::ScalarType>(ty[i]); };
    return {dx.view(ctx->saved_data["shape"].toIntVector()).to(dt(0)), dw.to(dt(1)), db.to(dt(2)), Tensor(),
            Tensor()};
  }
};

std::vector<Tensor> norm(const Tensor& x, const Tensor& w, const Tensor& b, double eps, bool residual) {
  return guarded([&] { return NormFn::apply(x, w, b, eps, residual); });
}

// ---------------------------------------------------------------- products

// C = A @ B (+ add, laid out as C)
void gemm(const Tensor& A, const Tensor& B, const Tensor& C, mvm_gemm_desc d, const Tensor& add = Tensor()) {
  c10::OptionalDeviceGuard guard(C.device());
  const int64_t nbytes = check(mvm_gemm_workspace_bytes(&d));
  Tensor ws;
  if (nbytes > 0) ws = workspace(nbytes, C);
  check(mvm_gemm_f32(&d, fp(A), fp(B), fp(add), fpm(C), ws.defined() ? ws.mutable_data_ptr() : nullptr,
                     static_cast<size_t>(nbytes), stream_of(C)));
}

mvm_gemm_desc gemm_desc(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc, bool a_km,
                        bool b_km) {
  mvm_gemm_desc d{};
  d.m = m; d.n = n; d.k = k; d.batch = 1;
  d.lda = lda; d.ldb = ldb; d.ldc = ldc;
  d.a_kmajor = a_km; d.b_kmajor = b_km;
  return d;
}

constexpr int64_t kMaxLd = int64_t{1} << 21;

// Values of the streamed operand from which a `stream` product (delta_raw's
// gradient times W_dt: every channel read once, a few columns out, hardly any
// arithmetic) is left to the BLAS library.  Measured us, here / library with
// its default picks, by MB streamed, at 128 to 3072 channels and 392 to 98304
// rows: 25 MB and less 4-15 / 17-19 everywhere; 50 MB: 128 channels 18.3 / 18.2,
// 768 18.3 / 18.6, 1536 21.3 / 20.1; 63-79 MB: 320 19.4 / 19.2, 768 26.1 / 20.7;
// 101 MB: 1536 32.3 / 28.1, 3072 62 / 40; 126-157 MB: 320 34.8 / 26.1, 768 38.6 /
// 35.0, 1536 48 / 53, 3072 66 / 76; 302 MB: 768 81 / 70, 1536 82 / 91, 3072 138 /
// 127.  (The forward product is slower here in 2 of those 65 cases: it stays.)
constexpr int64_t kStreamValues = 12 << 20;

// out[q] (+)= op(A[q]) @ op(B[q]) for float32 (batch, rows, cols) views; ta /
// tb transpose an operand.  The kernels take contiguous columns, operand rows
// that do not overlap, and 16-byte rows of an operand whose summed index is the
// contiguous one (from 32 summed values up); other operands (a parameter that
// is an expanded row, say), and `stream` products from kStreamValues, are torch's.
void batched(const Tensor& A, const Tensor& B, Tensor& out, bool ta, bool tb, bool accumulate, bool stream) {
  TORCH_CHECK(A.dim() == 3 && B.dim() == 3 && out.dim() == 3, "batched products take 3-D tensors");
  const int64_t q = A.size(0), m = A.size(ta ? 2 : 1), k = A.size(ta ? 1 : 2), n = B.size(tb ? 1 : 2);
  // (the kernels only see pointers: the checks torch's products would make)
  TORCH_CHECK(B.size(0) == q && B.size(tb ? 2 : 1) == k && out.sizes() == at::IntArrayRef({q, m, n}),
              "batched products of ", A.sizes(), " and ", B.sizes(), " into ", out.sizes(), " do not fit");
  check_device({&A, &B, &out});
  for (const Tensor* t : {&A, &B, static_cast<const Tensor*>(&out)})
    TORCH_CHECK(t->scalar_type() == at::kFloat, "batched products take float32; got ", t->scalar_type());
  auto rows16 = [](const Tensor& t) { return t.stride(1) % 4 == 0 && t.stride(0) % 4 == 0 && aligned16(t); };
  auto rows = [](const Tensor& t) { return t.stride(2) == 1 && t.stride(1) >= t.size(2) && t.stride(1) < kMaxLd; };
  const bool ok = rows(A) && rows(B) && out.stride(2) == 1 && (k < 32 || ((ta || rows16(A)) && (!tb || rows16(B)))) &&
                  !(stream && q * m * k >= kStreamValues);
  if (ok) {
    auto d = gemm_desc(m, n, k, A.stride(1), B.stride(1), out.stride(1), !ta, tb);
    d.batch = q;
    d.a_stride_batch = A.stride(0); d.b_stride_batch = B.stride(0); d.c_stride_batch = out.stride(0);
    gemm(A, B, out, d, accumulate ? out : Tensor());
    return;
  }
  const Tensor Av = ta ? A.transpose(1, 2) : A, Bv = tb ? B.transpose(1, 2) : B;
  if (accumulate)
    out.baddbmm_(Av, Bv);
  else
    at::bmm_out(out, Av, Bv);
}

// g with the layout and alignment the products take
Tensor dense(const Tensor& g) {
  const Tensor c = g.contiguous();
  return aligned16(c) ? c : c.clone();
}

// Whether the products take (x, W): float32 on the GPU outside autocast
// (whose casts at::linear applies), row lengths that are multiples of 4
// (16-byte rows) and below the kernels' limit, aligned weights.
bool usable(const Tensor& x, const Tensor& W, std::initializer_list<int64_t> widths) {
  bool ok = x.is_cuda() && x.device() == W.device() && x.scalar_type() == at::kFloat &&
            W.scalar_type() == at::kFloat && !at::autocast::is_autocast_enabled(at::kCUDA) && W.is_contiguous() &&
            aligned16(W);
  for (int64_t w : widths) ok = ok && w % 4 == 0 && w > 0 && w < kMaxLd;
  return ok;
}

// h (..., E) @ W (O, E)^T
struct InProjFn : Function<InProjFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h, const Tensor& W) {
    const int64_t O = W.size(0), E = W.size(1);
    const Tensor h2 = dense(h.reshape({-1, E}));
    const int64_t M = h2.size(0);
    auto shape = h.sizes().vec();
    ctx->saved_data["shape"] = shape;
    shape.back() = O;
    Tensor out = empty_like_opts(shape, h);  // (not a view: see OutProjFn)
    gemm(h2, W, out, gemm_desc(M, O, E, E, E, O, true, true));
    ctx->save_for_backward({h, W});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return grads(ctx, g); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor& W = sv[1];
    const int64_t O = W.size(0), E = W.size(1);
    Tensor dh, dW;
    // create_graph, or gradients batched by vmap (is_grads_batched): torch's
    // products, which have a derivative and a batching rule
    if (at::GradMode::is_enabled() || !g[0].has_storage()) {
      if (ctx->needs_input_grad(0)) dh = at::matmul(g[0], W);
      if (ctx->needs_input_grad(1)) dW = at::matmul(g[0].reshape({-1, O}).t(), sv[0].reshape({-1, E}));
      return {dh, dW};
    }
    const Tensor h2 = dense(sv[0].reshape({-1, E}));
    const int64_t M = h2.size(0);
    const Tensor g2 = dense(g[0].reshape({M, O}));
    if (ctx->needs_input_grad(0)) {
      dh = empty_like_opts({M, E}, g2);
      gemm(g2, W, dh, gemm_desc(M, E, O, O, E, E, true, false));
      dh = dh.view(ctx->saved_data["shape"].toIntVector());
    }
    if (ctx->needs_input_grad(1)) {
      dW = empty_like_opts({O, E}, g2);
      gemm(g2, h2, dW, gemm_desc(O, E, M, O, E, E, false, false));
    }
    return {dh, dW};
  }
};

// sum over k of y (..., K, D)[k] @ W (K, E, D)[k]^T: the K weight matrices
// are read where they lie, as one product over K * D, and their gradient
// comes out in the same layout, so no reordered copy of either is made.  A
// residual is added in the product's epilogue
struct OutProjFn : Function<OutProjFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& y, const Tensor& W, const OptTensor& res) {
    const int64_t K = W.size(0), E = W.size(1), D = W.size(2);
    const Tensor y2 = dense(y.reshape({-1, K * D}));
    const int64_t M = y2.size(0);
    // allocated in its final shape: a view made here could not be changed in place
    auto shape = y.sizes().vec();
    ctx->saved_data["shape"] = shape;
    shape.pop_back();
    shape.back() = E;
    Tensor out = empty_like_opts(shape, y);
    auto d = gemm_desc(M, E, K * D, K * D, D, E, true, true);
    if (K > 1) {
      d.b_seg = D;
      d.b_seg_stride = E * D;
    }
    gemm(y2, W, out, d, res.has_value() ? res->reshape({M, E}).contiguous() : Tensor());
    ctx->save_for_backward({y, W});
    ctx->saved_data["res"] = res.has_value();
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return grads(ctx, g); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor& W = sv[1];
    const int64_t K = W.size(0), E = W.size(1), D = W.size(2);
    Tensor dy, dW;
    const Tensor dres = ctx->saved_data["res"].toBool() ? g[0] : Tensor();
    if (at::GradMode::is_enabled() || !g[0].has_storage()) {  // as in InProjFn
      const Tensor Wc = W.permute({1, 0, 2}).reshape({E, K * D});
      if (ctx->needs_input_grad(0)) dy = at::matmul(g[0], Wc).view(ctx->saved_data["shape"].toIntVector());
      if (ctx->needs_input_grad(1))
        dW = at::matmul(g[0].reshape({-1, E}).t(), sv[0].reshape({-1, K * D})).view({E, K, D}).permute({1, 0, 2});
      return {dy, dW, dres};
    }
    const Tensor y2 = dense(sv[0].reshape({-1, K * D}));
    const int64_t M = y2.size(0);
    const Tensor g2 = dense(g[0].reshape({M, E}));
    if (ctx->needs_input_grad(0)) {
      dy = empty_like_opts({M, K, D}, g2);
      auto d = gemm_desc(M, D, E, E, D, K * D, true, false);
      d.batch = K;
      d.b_stride_batch = E * D;
      d.c_stride_batch = D;
      gemm(g2, W, dy, d);
      dy = dy.view(ctx->saved_data["shape"].toIntVector());
    }
    if (ctx->needs_input_grad(1)) {
      dW = empty_like_opts({K, E, D}, g2);
      auto d = gemm_desc(E, D, M, E, K * D, D, false, false);
      d.batch = K;
      d.b_stride_batch = D;
      d.c_stride_batch = E * D;
      gemm(g2, y2, dW, d);
    }
    return {dy, dW, dres};
  }
};

Tensor in_proj(const Tensor& h, const Tensor& W) {
  if (h.size(-1) == W.size(1) && usable(h, W, {W.size(0), W.size(1)})) return InProjFn::apply(h, W);
  return at::linear(h, W);
}

Tensor out_proj(const Tensor& y, const Tensor& W, const OptTensor& res) {
  const int64_t K = W.size(0), E = W.size(1), D = W.size(2);
  if (y.size(-1) == D && y.size(-2) == K && usable(y, W, {E, D, K * D}) && (K == 1 || D % 16 == 0)) {
    auto shape = y.sizes().vec();
    shape.pop_back();
    shape.back() = E;
    if (!res.has_value()) return OutProjFn::apply(y, W, res);
    if (res->scalar_type() == at::kFloat && res->device() == y.device() && res->sizes() == shape)
      return OutProjFn::apply(y, W, res);
    return *res + OutProjFn::apply(y, W, OptTensor());
  }
  // one product over the concatenated directions (a reordered copy of W)
  auto shape = y.sizes().vec();
  shape.pop_back();
  shape.back() = K * D;
  const Tensor out = at::linear(y.reshape(shape), W.permute({1, 0, 2}).reshape({E, K * D}));
  return res.has_value() ? *res + out : out;
}

// -------------------------------------------------------------- block core

// (buffers..., parameters...) -> the buffers, differentiable w.r.t. the
// parameters that are their slices: the backward hands each buffer's gradient
// to its K parameters as K contiguous slices
struct DirectionParamsFn : Function<DirectionParamsFn> {
  static variable_list forward(AutogradContext* ctx, at::TensorList bufs, at::TensorList params) {
    const int64_t K = bufs.empty() ? 0 : bufs[0].size(0);
    ctx->saved_data["nbuf"] = static_cast<int64_t>(bufs.size());
    ctx->saved_data["K"] = K;
    variable_list out;
    out.reserve(bufs.size());
    for (const Tensor& b : bufs) out.push_back(b.view_as(b));
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const int64_t nbuf = ctx->saved_data["nbuf"].toInt(), K = ctx->saved_data["K"].toInt();
    variable_list out(nbuf);
    for (const Tensor& g : grads) {
      if (g.defined()) {
        for (Tensor& s : g.contiguous().unbind(0)) out.push_back(std::move(s));
      } else {
        out.resize(out.size() + K);
      }
    }
    return out;
  }
};

std::vector<Tensor> direction_params(const std::vector<Tensor>& bufs, const std::vector<Tensor>& params) {
  return guarded([&] { return DirectionParamsFn::apply(at::TensorList(bufs), at::TensorList(params)); });
}

// whether params[i * K + k] is the k-th slice of bufs[i], for all of them
bool stacks_match(const std::vector<Tensor>& bufs, const std::vector<Tensor>& params) {
  if (bufs.empty() || params.size() % bufs.size() != 0) return false;
  const size_t K = params.size() / bufs.size();
  for (size_t i = 0; i < bufs.size(); ++i) {
    const Tensor& b = bufs[i];
    if (b.size(0) != static_cast<int64_t>(K)) return false;
    const char* base = static_cast<const char*>(b.const_data_ptr());
    const int64_t step = b.stride(0) * b.element_size();
    const auto shape = b.sizes().slice(1);
    for (size_t k = 0; k < K; ++k) {
      const Tensor& p = params[i * K + k];
      if (p.const_data_ptr() != base + static_cast<int64_t>(k) * step || p.scalar_type() != b.scalar_type() ||
          p.sizes() != shape || p.device() != b.device() || !p.is_contiguous())
        return false;
    }
  }
  return true;
}

// (B, N, K, X) view of a direction-major (K, B*N, X) tensor
Tensor bnkd(const Tensor& t, int64_t bsz, int64_t n) {
  return t.view({t.size(0), bsz, n, t.size(2)}).permute({1, 2, 0, 3});
}

// (K, rows, P) view whose rows are a multiple of 4 values apart: 16-byte
// rows for the products that read them
Tensor padded_rows(int64_t K, int64_t rows, int64_t P, const Tensor& like) {
  return empty_like_opts({K, rows, (P + 3) / 4 * 4}, like).narrow(2, 0, P);
}

// xz (B, N, K, 2*D_inner) from in_proj -> gated scan output (B, N, K, D_inner)
// (mamba_block.py:166-190, all K directions at once):
//   xc    = silu(causal depthwise conv(x) + conv_b)      along each scan order
//   dbc   = x_proj(xc)                                   (K, B*N, R + 2N)
//   delta = softplus(dt_proj(dbc[:R]) + dt_bias)         inside the scan, dt_proj
//           included up to rank 48 (d_model 768), and delta_raw written for the backward
//   y     = scan(xc, delta, -exp(A_log), B, C, D) * silu(z)
// The scan kernels take A_log and form A = -exp(A_log) themselves; their dA
// output is the gradient of A_log.  The backward writes the gradient of xz in
// place: the conv's dx and the gate's dz land in its two halves.
struct CoreFn : Function<CoreFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& xz, const Tensor& conv_w, const Tensor& conv_b,
                        const Tensor& W_x, const Tensor& W_dt, const Tensor& b_dt, const Tensor& A_log,
                        const Tensor& Dv, const OptTensor& tok_, int64_t chunk_len, bool save) {
    const Tensor tok = tok_.value_or(Tensor());
    const int64_t bsz = xz.size(0), n = xz.size(1), K = xz.size(2), din = xz.size(3) / 2;
    const int64_t R = W_dt.size(2), ns = A_log.size(2), M = bsz * n;
    check_device({&xz, &conv_w, &conv_b, &W_x, &W_dt, &b_dt, &A_log, &Dv});
    TORCH_CHECK(conv_w.size(0) == K && conv_w.size(1) == din && conv_b.sizes() == at::IntArrayRef({K, din}) &&
                    W_dt.sizes() == at::IntArrayRef({K, din, R}),
                "the block's conv ", conv_w.sizes(), ", ", conv_b.sizes(), " and dt_proj ", W_dt.sizes(),
                " do not fit K=", K, ", D_inner=", din);
    const Tensor xb = xz.narrow(3, 0, din), z = xz.narrow(3, din, din);
    Tensor xc = empty_like_opts({K, M, din}, xz);
    conv_fwd(xb, conv_w, conv_b, bnkd(xc, bsz, n), tok);                               // :170-171
    Tensor dbc = padded_rows(K, M, R + 2 * ns, xz);
    batched(xc, W_x, dbc, false, true, false, false);                                  // :174
    const Tensor bc = bnkd(dbc, bsz, n);
    // dt_proj (:180) inside the scan, up to its largest rank, else as a product
    // (which writes delta_raw for the scan to read: block steps of 4 x 6272
    // rows of 768 channels 1529 us inside, 1526 with the product; of 6 x 16384
    // rows 5985 and 6043; an encoder's forward of 8 x 1024 rows 1289 and 1314)
    const bool dt_in = R <= MVM_SCAN_MAX_DT_RANK && W_dt.is_contiguous();
    // (forward only: delta_raw is never formed in memory; xc lends its layout)
    Tensor delta_raw = dt_in && !save ? xc : empty_like_opts({K, M, din}, xz);
    if (!dt_in) batched(dbc.narrow(2, 0, R), W_dt, delta_raw, false, true, false, false);
    // (the products of a block round more than its scan does)
    if (chunk_len == 0) {
      const auto d = make_desc(bnkd(xc, bsz, n), bc.narrow(3, R, ns), at::kFloat, at::kFloat, tok, 0);
      chunk_len = check(mvm_scan_long_chunk_len(&d));
    }
    const auto o = fused_fwd(bnkd(xc, bsz, n), bnkd(delta_raw, bsz, n), b_dt, A_log, bc.narrow(3, R, ns),
                             bc.narrow(3, R + ns, ns), Dv, z, tok, chunk_len, save, true,
                             dt_in ? bc.narrow(3, 0, R) : Tensor(), W_dt);                  // :180-190
    if (save) {
      ctx->save_for_backward({xz, conv_w, conv_b, W_x, W_dt, b_dt, A_log, Dv, tok, xc, dbc, delta_raw, o.y_raw,
                              o.ckpt});
      ctx->saved_data["chunk"] = chunk_len;
    }
    return o.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&] { return once_differentiable(grads(ctx, g), g, "the Mamba block's core"); });
  }
  static variable_list grads(AutogradContext* ctx, const variable_list& grads) {
    const auto sv = ctx->get_saved_variables();
    // refused at once, except where dt_proj is frozen: there the first
    // derivative was always given, and once_differentiable refuses the second
    TORCH_CHECK(!(at::GradMode::is_enabled() && sv[4].requires_grad()),
                "the Mamba block's core is not twice differentiable (create_graph=True)");
    at::NoGradGuard no_grad;
    const Tensor &xz = sv[0], &conv_w = sv[1], &conv_b = sv[2], &W_x = sv[3], &W_dt = sv[4], &b_dt = sv[5],
                 &A_log = sv[6], &Dv = sv[7], &tok = sv[8], &xc = sv[9], &dbc = sv[10], &delta_raw = sv[11];
    const int64_t bsz = xz.size(0), n = xz.size(1), K = xz.size(2), din = xz.size(3) / 2;
    const int64_t R = W_dt.size(2), ns = A_log.size(2), M = bsz * n;
    Tensor dxz = empty_like_opts(xz.sizes(), xz);
    // (the strides of dbc, which a saved-tensor hook may have changed)
    Tensor d_dbc = dbc.stride(2) == 1 && dbc.stride(0) == M * dbc.stride(1)
                       ? empty_like_opts({K, M, dbc.stride(1)}, xz).narrow(2, 0, dbc.size(2))
                       : at::empty_strided(dbc.sizes(), dbc.strides(), xz.options().requires_grad(false));
    const Tensor bc = bnkd(dbc, bsz, n), g_bc = bnkd(d_dbc, bsz, n);
    Tensor du = at::empty_strided(xc.sizes(), xc.strides(), xc.options().requires_grad(false));
    Tensor ddelta_raw = at::empty_strided(delta_raw.sizes(), delta_raw.strides(),
                                          delta_raw.options().requires_grad(false));
    FusedGrads g;
    g.du = bnkd(du, bsz, n);
    g.ddelta_raw = bnkd(ddelta_raw, bsz, n);
    g.dB = g_bc.narrow(3, R, ns);
    g.dC = g_bc.narrow(3, R + ns, ns);
    g.dz = dxz.narrow(3, din, din);
    fused_bwd(bnkd(xc, bsz, n), bnkd(delta_raw, bsz, n), b_dt, A_log, bc.narrow(3, R, ns),
              bc.narrow(3, R + ns, ns), Dv, xz.narrow(3, din, din), sv[12], sv[13], grads[0], tok,
              ctx->saved_data["chunk"].toInt(), true, g);
    // dt_proj: delta_raw = dt @ W_dt^T; the product writes the first R
    // columns of d_dbc in place
    Tensor d_dt = d_dbc.narrow(2, 0, R);
    batched(ddelta_raw, W_dt, d_dt, false, false, false, true);
    Tensor dW_dt = empty_like_opts(W_dt.sizes(), xz);
    batched(ddelta_raw, dbc.narrow(2, 0, R), dW_dt, true, false, false, false);
    // x_proj: dbc = xc @ W_x^T; its input gradient is added to the scan's du
    batched(d_dbc, W_x, du, false, false, true, false);
    Tensor dW_x = empty_like_opts(W_x.sizes(), xz);
    batched(d_dbc, xc, dW_x, true, false, false, false);
    // conv + SiLU: dx lands in the first half of dxz
    auto [dconv_w, dconv_b] = conv_bwd(xz.narrow(3, 0, din), conv_w, conv_b, bnkd(du, bsz, n),
                                       dxz.narrow(3, 0, din), tok);
    return {dxz, dconv_w, dconv_b, dW_x, dW_dt, g.ddbias, g.dA, g.dD, Tensor(), Tensor(), Tensor()};
  }
};

// K MambaBlocks on one (B, N, E) input, block k scanning in the order of
// tok[k]; the sum of their outputs, and of the residual when there is one.  params: the nine kinds of
// mamba_block.STACKED_PARAMS, kind-major, K each; stacks: the buffers whose
// leading K slices they are (empty: a single block).
Tensor directional(const Tensor& h, const std::vector<Tensor>& params, const std::vector<Tensor>& stacks,
                   int64_t K, const OptTensor& tok_, int64_t chunk_len, bool detach, const OptTensor& res) {
  return guarded([&] {
    if (h.dim() != 3) bad_value("the block input must be (B, L, d_model); got " + shape_str(h));
    variable_list per;
    if (stacks.empty()) {
      for (const Tensor& p : params) per.push_back(p.unsqueeze(0));
    } else {
      std::vector<Tensor> bufs;
      for (const Tensor& s : stacks) bufs.push_back(s.size(0) == K ? s : s.narrow(0, 0, K));
      per = DirectionParamsFn::apply(at::TensorList(bufs), at::TensorList(params));
    }
    const int64_t bsz = h.size(0), n = h.size(1), E = per[0].size(2), din = per[0].size(1) / 2;
    const Tensor xz = in_proj(h, per[0].reshape({K * 2 * din, E})).view({bsz, n, K, 2 * din});  // :165-167
    const Tensor conv_w = per[1].reshape({K, din, per[1].size(-1)});
    variable_list args = {xz, conv_w, per[2], per[3], per[4], per[5], per[6], per[7]};
    bool needs = false;
    for (Tensor& t : args) {
      t = t.to(at::kFloat);
      if (detach) t = t.detach();
      needs = needs || t.requires_grad();
    }
    OptTensor tok;
    if (tok_.has_value()) tok = tok_->to(h.device()).contiguous();
    const bool save = !detach && at::GradMode::is_enabled() && needs;
    const Tensor y = CoreFn::apply(args[0], args[1], args[2], args[3], args[4], args[5], args[6], args[7], tok,
                                   chunk_len, save);                                          // :170-190
    return out_proj(y, per[8], res);                                                         // :191, :562-566
  });
}

Tensor batched_py(const Tensor& A, const Tensor& B, const OptTensor& out_, bool ta, bool tb, bool accumulate,
                  bool stream) {
  return guarded([&] {
    at::NoGradGuard no_grad;
    Tensor out = out_.has_value() ? *out_ : empty_like_opts({A.size(0), A.size(ta ? 2 : 1), B.size(tb ? 1 : 2)}, A);
    batched(A, B, out, ta, tb, accumulate, stream);
    return out;
  });
}

void set_timer(const py::object& start, const py::object& stop) {
  // kept for the life of the process: a launch may be using them
  if (!start.is_none() && g_timer_start == nullptr) {
    g_timer_start = new py::object(start);
    g_timer_stop = new py::object(stop);
  }
  g_timing.store(!start.is_none());
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("scan", &scan);
  m.def("scan_forward", &scan_forward);
  m.def("scan_backward", &scan_backward);
  m.def("scan_fused_forward", &scan_fused_forward);
  m.def("scan_fused_backward", &scan_fused_backward);
  m.def("conv_silu", &conv_silu);
  m.def("norm", &norm);
  m.def("in_proj", [](const Tensor& h, const Tensor& W) { return guarded([&] { return in_proj(h, W); }); });
  m.def("out_proj", [](const Tensor& y, const Tensor& W) { return guarded([&] { return out_proj(y, W, std::nullopt); }); });
  m.def("batched", &batched_py);
  m.def("direction_params", &direction_params);
  m.def("stacks_match", &stacks_match);
  m.def("directional", &directional);
  m.def("set_timer", &set_timer);
}
