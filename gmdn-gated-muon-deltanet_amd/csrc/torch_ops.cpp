// torch.ops.gmdn.*: the C-ABI entry points as torch operators, with autograd.
//
// Each operator wraps one call of libgmdn_scan.so (include/*.h) on the
// tensors' current stream; gmdn_amd/ops.py documents them and registers
// their shape-only fake implementations.  They live in C++ because a small
// training call is bound by the host: through Python operators and a Python
// backward run by autograd's device thread, one forward + backward of the
// fused core at B1 H2 T64 d64 took 260 us of host time; it takes 99 us here
// (the drop-in scan 206 -> 87 us, an inference call 30 -> 12 us).
//
// The autograd kernels sit at the Autograd dispatch key as torch's own
// autograd functions (saved tensors go through SavedVariable, so saved-tensor
// hooks apply), and call the operators through the dispatcher, so tracing,
// fake tensors and functionalisation see the same operators as before.  Each
// function's outputs are the differentiable ones only: what the forward saves
// (moments, checkpoints, 1 / rms) reaches the caller through a pointer, since
// compiled autograd takes no function with non-differentiable outputs.
#include "../../include/gmdn_front.h"
#include "../../include/gmdn_scan.h"
#include "../../include/gmdn_tail.h"

#include <ATen/ATen.h>
#include <algorithm>
#include <array>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <atomic>
#include <optional>
#include <tuple>
#include <type_traits>
#include <vector>

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
constexpr int64_t CHUNK = 64;

// The process's product precision (gmdn_amd.scan.set_precision), read by the
// muon core's backward.
std::atomic<int64_t> default_precision{GMDN_PREC_TF32};

void check(int rc, const char* what) {
  TORCH_CHECK(rc == GMDN_OK, what, " failed with code ", rc, ": ", gmdn_error_string(rc));
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
float* fp(const Tensor& t) { return t.numel() ? t.data_ptr<float>() : nullptr; }
const float* fp(const OptTensor& t) { return t ? t->data_ptr<float>() : nullptr; }
Tensor f32_empty(const Tensor& like, at::IntArrayRef size) { return at::empty(size, like.options().dtype(at::kFloat)); }
Tensor none_of(const Tensor& like) { return f32_empty(like, {0}); }
Tensor bytes_of(const Tensor& like, size_t n) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte));
}

void check_rank(const Tensor& t, int64_t rank, const char* what) {
  TORCH_CHECK(t.dim() == rank, what, " must have ", rank, " dimensions, got shape ", t.sizes());
}

// ------------------------------------------------------------ token streams
void check_tokens(const Tensor& q, const Tensor& k, const Tensor& v) {
  for (const Tensor* t : {&q, &k, &v}) {
    TORCH_CHECK(t->scalar_type() == at::kBFloat16 || t->scalar_type() == at::kFloat,
                "gmdn::chunk_fwd / chunk_bwd take bfloat16 or float32 q, k, v, got ", t->scalar_type());
    TORCH_CHECK(t->scalar_type() == q.scalar_type(), "q, k, v must share one dtype, got ", q.scalar_type(), " and ",
                t->scalar_type());
    TORCH_CHECK(t->dim() == 4, "token streams are (B, H, T, d), got shape ", t->sizes());
  }
}

// Whether t's elements fill its storage extent exactly once: the strides of a
// contiguous tensor with permuted dimensions (no zero strides, no gaps).
bool dense_permutation(const Tensor& t) {
  std::array<std::pair<int64_t, int64_t>, 4> d;
  int n = 0;
  for (int64_t i = 0; i < t.dim() && i < 4; ++i)
    if (t.size(i) != 1) d[n++] = {t.stride(i), t.size(i)};
  std::sort(d.begin(), d.begin() + n);
  int64_t want = 1;
  for (int i = 0; i < n; ++i) {
    if (d[i].first != want) return false;
    want *= d[i].second;
  }
  return true;
}
bool rows_fit(const Tensor& t) {
  return t.stride(-1) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0;
}
// Token stream with a unit-stride last dim, B/H/T strides in multiples of 8
// elements and a 16-byte-aligned base; `dense`: also a dense permutation (the
// backward writes each stream's gradient with the stream's own strides).
Tensor tok(const Tensor& t, bool dense = false) {
  if (!rows_fit(t) || (uintptr_t)t.data_ptr() % 16 || (dense && !dense_permutation(t)))
    return t.contiguous();
  return t;
}
// The strides of the output and gradient of token stream t: its own when they
// suit the kernels and t is a dense permutation, else contiguous.  The data
// pointer does not enter, so the fake implementations agree.
std::array<int64_t, 4> stream_strides(const Tensor& t) {
  std::array<int64_t, 4> s;
  if (rows_fit(t) && dense_permutation(t)) {
    std::copy(t.strides().begin(), t.strides().end(), s.begin());
  } else {
    s[3] = 1;
    for (int i = 2; i >= 0; --i) s[i] = s[i + 1] * std::max<int64_t>(t.size(i + 1), 1);
  }
  return s;
}
Tensor empty_like_stream(const Tensor& t) { return at::empty_strided(t.sizes(), stream_strides(t), t.options()); }
// x laid out with stream_strides(t) (a copy only when they differ)
Tensor as_stream_like(const Tensor& x, const Tensor& t) {
  if (x.strides() == at::IntArrayRef(stream_strides(t))) return x;
  return empty_like_stream(t).copy_(x);
}
Tensor gate(const Tensor& t) {
  Tensor c = t.to(at::kFloat).contiguous();
  return (uintptr_t)c.data_ptr() % 16 ? c.clone() : c;
}
OptTensor gate(const OptTensor& t) { return t ? OptTensor(gate(*t)) : OptTensor(); }

gmdn_chunk_desc chunk_desc(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, int64_t rule, int64_t ns,
                           double eps, int64_t precision) {
  gmdn_chunk_desc d{};
  d.B = q.size(0);
  d.H = q.size(1);
  d.T = q.size(2);
  d.d = (int32_t)q.size(3);
  d.C = CHUNK;
  d.rule = (int32_t)rule;
  d.ns = (int32_t)ns;
  d.dtype = q.scalar_type() == at::kFloat ? GMDN_DTYPE_F32 : GMDN_DTYPE_BF16;
  d.precision = (int32_t)precision;
  d.eps = (float)eps;
  for (int i = 0; i < 3; ++i) {
    d.sq[i] = q.stride(i);
    d.sk[i] = k.stride(i);
    d.sv[i] = v.stride(i);
    d.so[i] = o.stride(i);
  }
  return d;
}

// ------------------------------------------------------------------ the scan
std::tuple<Tensor, Tensor, Tensor> state_scan(const Tensor& U, const Tensor& K, const Tensor& a, const Tensor& b,
                                              const Tensor& m, const Tensor& n, int64_t rule, int64_t ns,
                                              int64_t precision, bool save_moments) {
  check_rank(U, 5, "U");
  const c10::DeviceGuard g(U.device());
  Tensor S = at::empty_like(U);
  Tensor M = rule != 0 && save_moments ? at::empty_like(U) : none_of(U);
  Tensor V = rule == 2 && save_moments ? at::empty_like(U) : none_of(U);
  check(gmdn_scan_fwd(fp(U), fp(K), fp(a), fp(b), fp(m), fp(n), fp(S), fp(M), fp(V), U.size(0) * U.size(1), U.size(2),
                      (int32_t)U.size(3), (int32_t)rule, (int32_t)ns, (int32_t)precision, stream_of(U)),
        "gmdn_scan_fwd");
  return {S, M, V};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> state_scan_bwd(
    const Tensor& U, const Tensor& K, const Tensor& a, const Tensor& b, const Tensor& m, const Tensor& n,
    const Tensor& S, const Tensor& M, const Tensor& V, const Tensor& gS_, int64_t rule, int64_t ns, int64_t precision) {
  check_rank(U, 5, "U");
  const c10::DeviceGuard g(U.device());
  Tensor gS = gS_.to(at::kFloat).contiguous();
  Tensor dU = at::empty_like(U), dK = at::empty_like(K);
  Tensor da = at::empty_like(a), db = at::empty_like(a), dm = at::empty_like(a), dn = at::empty_like(a);
  const int64_t BH = U.size(0) * U.size(1), N = U.size(2);
  const int32_t dh = (int32_t)U.size(3);
  const size_t ws_bytes = gmdn_scan_bwd_workspace_bytes(BH, N, dh, (int32_t)rule, (int32_t)ns);
  Tensor ws = ws_bytes ? bytes_of(U, ws_bytes) : Tensor();
  check(gmdn_scan_bwd(fp(U), fp(K), fp(a), fp(b), fp(m), fp(n), fp(S), fp(M), fp(V), fp(gS), fp(dU), fp(dK), fp(da),
                      fp(db), fp(dm), fp(dn), ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, BH, N, dh, (int32_t)rule,
                      (int32_t)ns, (int32_t)precision, stream_of(U)),
        "gmdn_scan_bwd");
  return {dU, dK, da, db, dm, dn};
}

// ------------------------------------------------------------ the fused core
// The chunk states are written for a backward, and always where the output
// kernel reads them (muon; float32 streams).
bool keeps_states(const Tensor& q, int64_t rule, bool record) {
  return record || rule == 1 || q.scalar_type() == at::kFloat;
}

std::tuple<Tensor, Tensor> chunk_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                                     const Tensor& g, const OptTensor& gmu, const OptTensor& gnu, int64_t rule,
                                     int64_t ns, double eps, bool record) {
  check_tokens(q, k, v);
  const c10::DeviceGuard guard(q.device());
  Tensor qc = tok(q), kc = tok(k), vc = tok(v), bc = gate(beta), gc = gate(g);
  OptTensor mc = gate(gmu), nc = gate(gnu);
  // o takes q's layout (the mixer's (B, T, H, d) storage, so that the head
  // norm and output projection read it without a transposing copy)
  Tensor o = empty_like_stream(q);
  const gmdn_chunk_desc desc = chunk_desc(qc, kc, vc, o, rule, ns, eps, GMDN_PREC_TF32);
  const bool keep = keeps_states(q, rule, record);
  Tensor states = keep ? f32_empty(q, {(int64_t)(gmdn_chunk_states_bytes(&desc) / 4)}) : none_of(q);
  check(gmdn_chunk_fwd(&desc, qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), fp(bc), fp(gc), fp(mc), fp(nc), o.data_ptr(),
                       keep ? states.data_ptr() : nullptr, stream_of(q)),
        "gmdn_chunk_fwd");
  return {o, states};
}

using Grads7 = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
Grads7 chunk_bwd_call(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta, const Tensor& g,
                      const OptTensor& gmu, const OptTensor& gnu, const Tensor& states, const Tensor& dO, int64_t rule,
                      int64_t ns, double eps, int64_t precision) {
  check_tokens(q, k, v);
  const c10::DeviceGuard guard(q.device());
  Tensor qc = tok(q, true), kc = tok(k, true), vc = tok(v, true), bc = gate(beta), gc = gate(g);
  OptTensor mc = gate(gmu), nc = gate(gnu);
  Tensor dOc = tok(dO.to(q.scalar_type()));
  // the kernels write dq, dk, dv with the strides of q, k, v (dense here)
  Tensor dq = at::empty_strided(qc.sizes(), qc.strides(), qc.options()),
         dk = at::empty_strided(kc.sizes(), kc.strides(), kc.options()),
         dv = at::empty_strided(vc.sizes(), vc.strides(), vc.options());
  Tensor dbeta = at::empty_like(bc), dg = at::empty_like(gc);
  Tensor dgmu = mc ? at::empty_like(*mc) : none_of(q), dgnu = nc ? at::empty_like(*nc) : none_of(q);
  const gmdn_chunk_desc desc = chunk_desc(qc, kc, vc, dOc, rule, ns, eps, precision);
  const size_t ws_bytes = gmdn_chunk_bwd_workspace_bytes(&desc);
  Tensor ws = ws_bytes ? bytes_of(q, ws_bytes) : Tensor();
  check(gmdn_chunk_bwd(&desc, qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), fp(bc), fp(gc), fp(mc), fp(nc),
                       states.data_ptr(), dOc.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), fp(dbeta), fp(dg),
                       mc ? fp(dgmu) : nullptr, nc ? fp(dgnu) : nullptr, ws_bytes ? ws.data_ptr() : nullptr, ws_bytes,
                       stream_of(q)),
        "gmdn_chunk_bwd");
  // the fake implementation cannot see data pointers: a stream that tok
  // copied gets its gradient back in the strides the fake reports
  return {as_stream_like(dq, q), as_stream_like(dk, k), as_stream_like(dv, v), dbeta, dg, dgmu, dgnu};
}
Grads7 chunk_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta, const Tensor& g,
                 const OptTensor& gmu, const OptTensor& gnu, const Tensor& states, const Tensor& dO, int64_t rule,
                 int64_t ns, double eps) {
  return chunk_bwd_call(q, k, v, beta, g, gmu, gnu, states, dO, rule, ns, eps, GMDN_PREC_TF32);
}
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> chunk_bwd_muon(const Tensor& q, const Tensor& k,
                                                                          const Tensor& v, const Tensor& beta,
                                                                          const Tensor& g, const Tensor& gmu,
                                                                          const Tensor& states, const Tensor& dO,
                                                                          int64_t ns, int64_t precision) {
  auto [dq, dk, dv, db, dg, dm, dn] = chunk_bwd_call(q, k, v, beta, g, gmu, OptTensor(), states, dO, 1, ns, 1e-6, precision);
  return {dq, dk, dv, db.to(beta.scalar_type()), dg.to(g.scalar_type()), dm.to(gmu.scalar_type())};
}

// ------------------------------------------------------- the token-exact mode
int64_t wy_ckpt_floats(const gmdn_chunk_desc& desc) {
  return std::max<int64_t>((int64_t)gmdn_wy_fwd_workspace_bytes(&desc) / 4, 4);
}
std::tuple<Tensor, Tensor> wy_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                                  const Tensor& g, bool record) {
  check_tokens(q, k, v);
  const c10::DeviceGuard guard(q.device());
  Tensor qc = tok(q), kc = tok(k), vc = tok(v), bc = gate(beta), gc = gate(g), o = empty_like_stream(q);
  const gmdn_chunk_desc desc = chunk_desc(qc, kc, vc, o, 0, 0, 1e-6, GMDN_PREC_TF32);
  // the forward's workspace is the backward's checkpoint
  Tensor ws = f32_empty(q, {wy_ckpt_floats(desc)});
  check(gmdn_wy_fwd(&desc, qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), fp(bc), fp(gc), o.data_ptr(), ws.data_ptr(),
                    (size_t)ws.numel() * 4, stream_of(q)),
        "gmdn_wy_fwd");
  return {o, record ? ws : none_of(q)};
}
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> wy_bwd(const Tensor& q, const Tensor& k, const Tensor& v,
                                                          const Tensor& beta, const Tensor& g, const Tensor& ckpt,
                                                          const Tensor& dO) {
  check_tokens(q, k, v);
  const c10::DeviceGuard guard(q.device());
  Tensor qc = tok(q, true), kc = tok(k, true), vc = tok(v, true), bc = gate(beta), gc = gate(g);
  Tensor dOc = tok(dO.to(q.scalar_type()));
  Tensor dq = at::empty_strided(qc.sizes(), qc.strides(), qc.options()),
         dk = at::empty_strided(kc.sizes(), kc.strides(), kc.options()),
         dv = at::empty_strided(vc.sizes(), vc.strides(), vc.options());
  Tensor dbeta = at::empty_like(bc), dg = at::empty_like(gc);
  const gmdn_chunk_desc desc = chunk_desc(qc, kc, vc, dOc, 0, 0, 1e-6, GMDN_PREC_TF32);
  const size_t ws_bytes = std::max<size_t>(gmdn_wy_bwd_workspace_bytes(&desc), 16);
  Tensor ws = bytes_of(q, ws_bytes);
  check(gmdn_wy_bwd(&desc, qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), fp(bc), fp(gc), ckpt.data_ptr(), dOc.data_ptr(),
                    dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), fp(dbeta), fp(dg), ws.data_ptr(), ws_bytes,
                    stream_of(q)),
        "gmdn_wy_bwd");
  return {as_stream_like(dq, q), as_stream_like(dk, k), as_stream_like(dv, v), dbeta, dg};
}

// ------------------------------------------------------- the mixer's front and tail
int32_t dtype_code(const Tensor& t) {
  TORCH_CHECK(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat,
              "the mixer front-end kernels take bfloat16 or float32, got ", t.scalar_type());
  return t.scalar_type() == at::kFloat ? GMDN_DTYPE_F32 : GMDN_DTYPE_BF16;
}

std::tuple<Tensor, Tensor, Tensor> front_fwd(const Tensor& y, const Tensor& weight, const Tensor& bias, int64_t dh) {
  check_rank(y, 3, "y");
  const c10::DeviceGuard guard(y.device());
  const int64_t B = y.size(0), T = y.size(1), C3 = y.size(2), D = C3 / 3, K = weight.size(-1);
  Tensor yc = y.contiguous(), w = weight.reshape({C3, K}).to(at::kFloat).contiguous(),
         bc = bias.to(at::kFloat).contiguous();
  Tensor q = at::empty({B, T, D}, y.options()), k = at::empty({B, T, D}, y.options()),
         v = at::empty({B, T, D}, y.options());
  check(gmdn_front_fwd(yc.data_ptr(), fp(w), fp(bc), q.data_ptr(), k.data_ptr(), v.data_ptr(), B, T, (int32_t)D,
                       (int32_t)dh, (int32_t)K, dtype_code(y), stream_of(y)),
        "gmdn_front_fwd");
  return {q, k, v};
}
std::tuple<Tensor, Tensor, Tensor> front_bwd(const Tensor& y, const Tensor& weight, const Tensor& bias,
                                             const Tensor& dq, const Tensor& dk, const Tensor& dv, int64_t dh) {
  check_rank(y, 3, "y");
  const c10::DeviceGuard guard(y.device());
  const int64_t B = y.size(0), T = y.size(1), C3 = y.size(2), D = C3 / 3, K = weight.size(-1);
  Tensor yc = y.contiguous(), w = weight.reshape({C3, K}).to(at::kFloat).contiguous(),
         bc = bias.to(at::kFloat).contiguous();
  Tensor gq = dq.to(y.scalar_type()).contiguous(), gk = dk.to(y.scalar_type()).contiguous(),
         gv = dv.to(y.scalar_type()).contiguous();
  Tensor dy = at::empty_like(yc);
  Tensor partial = f32_empty(y, {(int64_t)gmdn_front_bwd_workspace_floats(B, T, (int32_t)D, (int32_t)K)});
  check(gmdn_front_bwd(yc.data_ptr(), fp(w), fp(bc), gq.data_ptr(), gk.data_ptr(), gv.data_ptr(), dy.data_ptr(),
                       fp(partial), B, T, (int32_t)D, (int32_t)dh, (int32_t)K, dtype_code(y), stream_of(y)),
        "gmdn_front_bwd");
  Tensor sums = partial.view({-1, C3, K + 1}).sum(0);
  return {dy, sums.narrow(1, 0, K).reshape(weight.sizes()).to(weight.scalar_type()),
          sums.select(1, K).to(bias.scalar_type()).contiguous()};
}

Tensor gates_fwd(const Tensor& y, int64_t heads, int64_t n_gates) {
  check_rank(y, 3, "y");
  const c10::DeviceGuard guard(y.device());
  Tensor yc = y.contiguous(), out = f32_empty(y, {n_gates, y.size(0), heads, y.size(1)});
  check(gmdn_gates_fwd(yc.data_ptr(), fp(out), y.size(0), y.size(1), (int32_t)heads, (int32_t)n_gates, dtype_code(yc),
                       stream_of(y)),
        "gmdn_gates_fwd");
  return out;
}
Tensor gates_bwd(const Tensor& y, const Tensor& dout, int64_t heads, int64_t n_gates) {
  check_rank(y, 3, "y");
  const c10::DeviceGuard guard(y.device());
  Tensor yc = y.contiguous(), dc = dout.to(at::kFloat).contiguous(), dy = at::empty_like(yc);
  check(gmdn_gates_bwd(yc.data_ptr(), fp(dc), dy.data_ptr(), y.size(0), y.size(1), (int32_t)heads, (int32_t)n_gates,
                       dtype_code(yc), stream_of(y)),
        "gmdn_gates_bwd");
  return dy;
}

std::tuple<Tensor, Tensor> head_norm_fwd(const Tensor& x, const Tensor& weight, double eps) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1);
  Tensor xc = x.contiguous(), wc = weight.contiguous(), out = at::empty_like(xc);
  Tensor rstd = f32_empty(x, xc.sizes().slice(0, xc.dim() - 1));
  check(gmdn_head_norm_fwd(xc.data_ptr(), fp(wc), out.data_ptr(), fp(rstd), d ? xc.numel() / d : 0, (int32_t)d,
                           (float)eps, dtype_code(xc), stream_of(x)),
        "gmdn_head_norm_fwd");
  return {out, rstd};
}
std::tuple<Tensor, Tensor> head_norm_bwd(const Tensor& x, const Tensor& weight, const Tensor& rstd,
                                         const Tensor& dout) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1);
  TORCH_CHECK(d > 0, "head_norm_bwd: rows of x are empty, shape ", x.sizes());
  Tensor xc = x.contiguous(), wc = weight.contiguous(), rc = rstd.contiguous();
  const int64_t rows = xc.numel() / d;
  Tensor dc = dout.to(x.scalar_type()).contiguous(), dx = at::empty_like(xc), dw = f32_empty(x, {d});
  Tensor ws = f32_empty(x, {std::max<int64_t>((int64_t)gmdn_head_norm_bwd_workspace_floats(rows, (int32_t)d), 1)});
  check(gmdn_head_norm_bwd(xc.data_ptr(), fp(wc), fp(rc), dc.data_ptr(), dx.data_ptr(), fp(dw), fp(ws),
                           (size_t)ws.numel(), rows, (int32_t)d, dtype_code(xc), stream_of(x)),
        "gmdn_head_norm_bwd");
  return {dx, dw};
}

// ------------------------------------------------------------------ autograd
// Calls through the dispatcher, below autograd.
template <class F>
auto op(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}
// A kernel's signature with symbolic integers: a traced size reaches the
// schema unspecialised, and only the kernels themselves see plain integers.
template <class F>
struct Symbolic;
template <class R, class... A>
struct Symbolic<R(A...)> {
  using T = R(std::conditional_t<std::is_same_v<A, int64_t>, c10::SymInt, A>...);
};
#define GMDN_OP(fn) \
  ([]() -> const auto& { static const auto h = op<Symbolic<decltype(fn)>::T>("gmdn::" #fn); return h; }())

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
Tensor opt(const OptTensor& t) { return t ? *t : Tensor(); }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

struct StateScan : torch::autograd::Function<StateScan> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& U, const Tensor& K, const Tensor& a, const Tensor& b,
                        const Tensor& m, const Tensor& n, c10::SymInt rule, c10::SymInt ns, c10::SymInt precision,
                        bool save, std::pair<Tensor, Tensor>* moments) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [S, M, V] = GMDN_OP(state_scan).call(U, K, a, b, m, n, rule, ns, precision, save);
    *moments = {M, V};
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({U, K, a, b, m, n, S, M, V});
    ctx->saved_data["rule"] = rule;
    ctx->saved_data["ns"] = ns;
    ctx->saved_data["precision"] = precision;
    return S;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor gS = grads[0].defined() ? grads[0] : at::zeros_like(s[6]);
    auto [dU, dK, da, db, dm, dn] = GMDN_OP(state_scan_bwd)
                                        .call(s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], gS,
                                              ctx->saved_data["rule"].toSymInt(), ctx->saved_data["ns"].toSymInt(),
                                              ctx->saved_data["precision"].toSymInt());
    return {dU, dK, da, db, dm, dn, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
std::tuple<Tensor, Tensor, Tensor> state_scan_ad(const Tensor& U, const Tensor& K, const Tensor& a, const Tensor& b,
                                                 const Tensor& m, const Tensor& n, c10::SymInt rule, c10::SymInt ns,
                                                 c10::SymInt precision, bool save) {
  if (!wants_grad({&U, &K, &a, &b, &m, &n})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(state_scan).call(U, K, a, b, m, n, rule, ns, precision, save);
  }
  std::pair<Tensor, Tensor> moments;
  Tensor S = StateScan::apply(U, K, a, b, m, n, rule, ns, precision, save, &moments);
  return {S, moments.first, moments.second};
}

struct ChunkFwd : torch::autograd::Function<ChunkFwd> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                        const Tensor& g, const OptTensor& gmu, const OptTensor& gnu, c10::SymInt rule, c10::SymInt ns,
                        double eps, bool record, Tensor* checkpoint) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [o, states] = GMDN_OP(chunk_fwd).call(q, k, v, beta, g, gmu, gnu, rule, ns, eps, record);
    *checkpoint = states;
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, beta, g, opt(gmu), opt(gnu), states});
    ctx->saved_data["rule"] = rule;
    ctx->saved_data["ns"] = ns;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["record"] = record;
    // a compiled backward is kept for its saved data: another setting, another trace
    ctx->saved_data["ieee"] = default_precision.load() == GMDN_PREC_IEEE;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    TORCH_CHECK(ctx->saved_data["record"].toBool(),
                "gmdn::chunk_fwd ran without recording its state checkpoint "
                "(grad mode was off at the call); it has no backward");
    const auto s = ctx->get_saved_variables();
    const Tensor dO = grads[0].defined() ? grads[0] : at::zeros_like(s[0]);
    const c10::SymInt rule = ctx->saved_data["rule"].toSymInt(), ns = ctx->saved_data["ns"].toSymInt();
    const Tensor none;
    if (rule == 1) {
      auto [dq, dk, dv, db, dg, dm] =
          GMDN_OP(chunk_bwd_muon).call(s[0], s[1], s[2], s[3], s[4], s[5], s[7], dO, ns, default_precision.load());
      return {dq, dk, dv, db, dg, dm, none, none, none, none, none, none};
    }
    auto [dq, dk, dv, db, dg, dm, dn] = GMDN_OP(chunk_bwd)
                                            .call(s[0], s[1], s[2], s[3], s[4], opt(s[5]), opt(s[6]), s[7], dO, rule, ns,
                                                  ctx->saved_data["eps"].toDouble());
    return {dq, dk, dv, db, dg, s[5].defined() ? dm : none, s[6].defined() ? dn : none, none, none, none, none, none};
  }
};
std::tuple<Tensor, Tensor> chunk_fwd_ad(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                                        const Tensor& g, const OptTensor& gmu, const OptTensor& gnu, c10::SymInt rule,
                                        c10::SymInt ns, double eps, bool record) {
  const Tensor m = opt(gmu), n = opt(gnu);
  if (!wants_grad({&q, &k, &v, &beta, &g, &m, &n})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(chunk_fwd).call(q, k, v, beta, g, gmu, gnu, rule, ns, eps, record);
  }
  Tensor states, o = ChunkFwd::apply(q, k, v, beta, g, gmu, gnu, rule, ns, eps, record, &states);
  return {o, states};
}

struct WyFwd : torch::autograd::Function<WyFwd> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                        const Tensor& g, bool record, Tensor* checkpoint) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [o, ckpt] = GMDN_OP(wy_fwd).call(q, k, v, beta, g, record);
    *checkpoint = ckpt;
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, beta, g, ckpt});
    ctx->saved_data["record"] = record;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    TORCH_CHECK(ctx->saved_data["record"].toBool(),
                "gmdn::wy_fwd ran without its checkpoint (grad mode was off at the call); it has no backward");
    const auto s = ctx->get_saved_variables();
    const Tensor dO = grads[0].defined() ? grads[0] : at::zeros_like(s[0]);
    auto [dq, dk, dv, db, dg] = GMDN_OP(wy_bwd).call(s[0], s[1], s[2], s[3], s[4], s[5], dO);
    return {dq, dk, dv, db.to(s[3].scalar_type()), dg.to(s[4].scalar_type()), Tensor(), Tensor()};
  }
};
std::tuple<Tensor, Tensor> wy_fwd_ad(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& beta,
                                     const Tensor& g, bool record) {
  if (!wants_grad({&q, &k, &v, &beta, &g})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(wy_fwd).call(q, k, v, beta, g, record);
  }
  Tensor ckpt, o = WyFwd::apply(q, k, v, beta, g, record, &ckpt);
  return {o, ckpt};
}

struct FrontFwd : torch::autograd::Function<FrontFwd> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, const Tensor& y, const Tensor& weight, const Tensor& bias,
                               c10::SymInt dh) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [q, k, v] = GMDN_OP(front_fwd).call(y, weight, bias, dh);
    ctx->save_for_backward({y, weight, bias});
    ctx->saved_data["dh"] = dh;
    return {q, k, v};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    auto [dy, dw, db] =
        GMDN_OP(front_bwd).call(s[0], s[1], s[2], g[0], g[1], g[2], ctx->saved_data["dh"].toSymInt());
    return {dy, dw, db, Tensor()};
  }
};
std::tuple<Tensor, Tensor, Tensor> front_fwd_ad(const Tensor& y, const Tensor& weight, const Tensor& bias,
                                                c10::SymInt dh) {
  if (!wants_grad({&y, &weight, &bias})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(front_fwd).call(y, weight, bias, dh);
  }
  auto r = FrontFwd::apply(y, weight, bias, dh);
  return {r[0], r[1], r[2]};
}

struct GatesFwd : torch::autograd::Function<GatesFwd> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& y, c10::SymInt heads, c10::SymInt n_gates) {
    at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({y});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["n_gates"] = n_gates;
    return GMDN_OP(gates_fwd).call(y, heads, n_gates);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    return {GMDN_OP(gates_bwd).call(s[0], g[0], ctx->saved_data["heads"].toSymInt(), ctx->saved_data["n_gates"].toSymInt()),
            Tensor(), Tensor()};
  }
};
Tensor gates_fwd_ad(const Tensor& y, c10::SymInt heads, c10::SymInt n_gates) {
  if (!wants_grad({&y})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(gates_fwd).call(y, heads, n_gates);
  }
  return GatesFwd::apply(y, heads, n_gates);
}

struct HeadNorm : torch::autograd::Function<HeadNorm> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, double eps, Tensor* rms) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [out, rstd] = GMDN_OP(head_norm_fwd).call(x, weight, eps);
    *rms = rstd;
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({x, weight, rstd});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = GMDN_OP(head_norm_bwd).call(s[0], s[1], s[2], g[0]);
    return {dx, dw, Tensor(), Tensor()};
  }
};
std::tuple<Tensor, Tensor> head_norm_fwd_ad(const Tensor& x, const Tensor& weight, double eps) {
  if (!wants_grad({&x, &weight})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return GMDN_OP(head_norm_fwd).call(x, weight, eps);
  }
  Tensor rstd, out = HeadNorm::apply(x, weight, eps, &rstd);
  return {out, rstd};
}

}  // namespace

extern "C" __attribute__((visibility("default"))) void gmdn_ops_set_precision(int64_t precision) {
  default_precision.store(precision);
}

TORCH_LIBRARY_FRAGMENT(gmdn, m) {
  const std::vector<at::Tag> PT2{at::Tag::pt2_compliant_tag};
  m.def("state_scan(Tensor U, Tensor K, Tensor a, Tensor b, Tensor m, Tensor n, SymInt rule, SymInt ns, "
        "SymInt precision, bool save_moments) -> (Tensor, Tensor, Tensor)", PT2);
  m.def("state_scan_bwd(Tensor U, Tensor K, Tensor a, Tensor b, Tensor m, Tensor n, Tensor S_all, Tensor M_all, "
        "Tensor V_all, Tensor gS, SymInt rule, SymInt ns, SymInt precision) -> "
        "(Tensor, Tensor, Tensor, Tensor, Tensor, Tensor)", PT2);
  m.def("chunk_fwd(Tensor q, Tensor k, Tensor v, Tensor beta, Tensor g, Tensor? gmu, Tensor? gnu, SymInt rule, "
        "SymInt ns, float eps, bool record) -> (Tensor, Tensor)", PT2);
  m.def("chunk_bwd(Tensor q, Tensor k, Tensor v, Tensor beta, Tensor g, Tensor? gmu, Tensor? gnu, Tensor states, "
        "Tensor dO, SymInt rule, SymInt ns, float eps) -> (Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor)", PT2);
  m.def("chunk_bwd_muon(Tensor q, Tensor k, Tensor v, Tensor beta, Tensor g, Tensor gmu, Tensor states, Tensor dO, "
        "SymInt ns, SymInt precision) -> (Tensor, Tensor, Tensor, Tensor, Tensor, Tensor)", PT2);
  m.def("wy_fwd(Tensor q, Tensor k, Tensor v, Tensor beta, Tensor g, bool record) -> (Tensor, Tensor)", PT2);
  m.def("wy_bwd(Tensor q, Tensor k, Tensor v, Tensor beta, Tensor g, Tensor ckpt, Tensor dO) -> "
        "(Tensor, Tensor, Tensor, Tensor, Tensor)", PT2);
  m.def("front_fwd(Tensor y, Tensor weight, Tensor bias, SymInt dh) -> (Tensor, Tensor, Tensor)", PT2);
  m.def("front_bwd(Tensor y, Tensor weight, Tensor bias, Tensor dq, Tensor dk, Tensor dv, SymInt dh) -> "
        "(Tensor, Tensor, Tensor)", PT2);
  m.def("gates_fwd(Tensor y, SymInt heads, SymInt n_gates) -> Tensor", PT2);
  m.def("gates_bwd(Tensor y, Tensor dout, SymInt heads, SymInt n_gates) -> Tensor", PT2);
  m.def("head_norm_fwd(Tensor x, Tensor weight, float eps) -> (Tensor, Tensor)", PT2);
  m.def("head_norm_bwd(Tensor x, Tensor weight, Tensor rstd, Tensor dout) -> (Tensor, Tensor)", PT2);
}

TORCH_LIBRARY_IMPL(gmdn, CUDA, m) {
  m.impl("state_scan", state_scan);
  m.impl("state_scan_bwd", state_scan_bwd);
  m.impl("chunk_fwd", chunk_fwd);
  m.impl("chunk_bwd", chunk_bwd);
  m.impl("chunk_bwd_muon", chunk_bwd_muon);
  m.impl("wy_fwd", wy_fwd);
  m.impl("wy_bwd", wy_bwd);
  m.impl("front_fwd", front_fwd);
  m.impl("front_bwd", front_bwd);
  m.impl("gates_fwd", gates_fwd);
  m.impl("gates_bwd", gates_bwd);
  m.impl("head_norm_fwd", head_norm_fwd);
  m.impl("head_norm_bwd", head_norm_bwd);
}

TORCH_LIBRARY_IMPL(gmdn, Autograd, m) {
  m.impl("state_scan", state_scan_ad);
  m.impl("chunk_fwd", chunk_fwd_ad);
  m.impl("wy_fwd", wy_fwd_ad);
  m.impl("front_fwd", front_fwd_ad);
  m.impl("gates_fwd", gates_fwd_ad);
  m.impl("head_norm_fwd", head_norm_fwd_ad);
  // The backward operators have no derivative: differentiating a gradient
  // taken with create_graph=True raises (unregistered, it would only warn and
  // drop the operator's terms).
  for (const char* name : {"state_scan_bwd", "chunk_bwd", "chunk_bwd_muon", "wy_bwd", "front_bwd", "gates_bwd",
                           "head_norm_bwd"})
    m.impl(name, torch::autograd::autogradNotImplementedFallback());
}
