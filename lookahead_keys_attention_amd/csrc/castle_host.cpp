// Host layer between PyTorch and the C ABI of libcastle_hip.so: the registered operators
// (torch.ops.castle_hip.*) with their autograd formulas, and the cached single-token step of a layer.
//
// This code is what stands between a call and its kernels, so it decides the time of every call whose
// kernels take less than about a third of a millisecond.  The same operators written in Python
// (torch.library.custom_op, autograd formulas, ctypes views) took 70 us of host time for a forward and
// 150 us more for a backward pass, a cached step 71 us; here an operator costs its allocations and launches.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <optional>
#include <tuple>
#include <vector>

#include "../../include/castle_hip.h"

namespace {

using at::Tensor;

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return CASTLE_F32;
    case at::kBFloat16: return CASTLE_BF16;
    case at::kHalf: return CASTLE_F16;
    default: TORCH_CHECK_TYPE(false, "castle HIP kernels support float32, bfloat16 and float16, not ", t.scalar_type());
  }
}

int64_t check(int64_t code, const char* what) {
  TORCH_CHECK(code >= 0, what, " failed: ", castle_error_string((int)code), " (code ", code, ")");
  return code;
}

void check_dims(int64_t d, const Tensor& t) {
  TORCH_CHECK_VALUE(d == 16 || d == 32 || d == 64 || d == 128,
                    "dim_head must be one of (16, 32, 64, 128) for the HIP kernels, got ", d);
  TORCH_CHECK_VALUE(t.scalar_type() != at::kFloat || d <= 64, "float32 HIP kernels support dim_head <= 64");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

castle_view4 view4(const Tensor& t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// the kernels read 16 bytes at a time along d; anything else is copied
Tensor readable(const Tensor& t) {
  const int64_t q = 16 / t.element_size();
  if (t.stride(3) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && t.stride(0) % q == 0 && t.stride(1) % q == 0 &&
      t.stride(2) % q == 0)
    return t;
  return t.contiguous();
}
Tensor packed_readable(const Tensor& t) {
  return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.contiguous();
}

// The kernels have no formula for a tangent (forward-mode derivatives); a result without one would stand for a derivative of zero.
void no_tangent(const Tensor& t) {
  TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(0).defined(), "the CASTLE kernels have no forward-mode derivatives (Castle(use_triton=False) has)");
}

Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

struct Shape {
  int B, H, L, d, dtype;
};

// part `i` of six of a packed (B, L, 6 H d) tensor, or the merged (B, L, H d) one (parts = 1), as a (B, H, L, d) view
castle_view4 packed_view(const Tensor& t, const Shape& s, int parts, int i) {
  const int64_t width = (int64_t)parts * s.H * s.d;
  return {static_cast<char*>(t.data_ptr()) + (int64_t)i * s.H * s.d * t.element_size(), s.L * width, s.d, width};
}

// six: qc, kc, vc, qu, ku, vu.  Returns what the backward pass needs back: (workspace, state), the state
// empty when it is not kept.
std::tuple<Tensor, Tensor> run_fwd(const castle_view4 (&six)[6], const Shape& s, double scale, int64_t flags, const castle_view4& out,
                                   const castle_view4& U, bool keep_state, const Tensor& like, const Tensor& prepared = Tensor()) {
  // prepared: a workspace that holds the partial maxima of |vu| already
  const int64_t nbytes = check(castle_fwd_workspace_bytes(s.B, s.H, s.L, s.d, s.dtype), "castle_fwd_workspace_bytes");
  const int64_t sbytes = check(castle_fwd_state_bytes(s.B, s.H, s.L, s.d, s.dtype), "castle_fwd_state_bytes");
  Tensor ws = prepared.defined() ? prepared : bytes(nbytes, like), state = bytes(sbytes, like);
  if (prepared.defined()) flags |= CASTLE_FLAG_AMAX_READY;
  check(castle_fwd(&six[0], &six[1], &six[2], &six[3], &six[4], &six[5], s.B, s.H, s.L, s.d, s.dtype, (float)scale, (int)flags, &out,
                   &U, ws.data_ptr(), nbytes, state.data_ptr(), sbytes, stream_of(like)),
        "castle_fwd");
  if (!keep_state) state = bytes(0, like);   // the caching allocator keeps the block until the stream is done with it
  return {ws, state};
}

int bwd_flags(int64_t flags, const Tensor& state) {
  return ((int)flags & ~CASTLE_FLAG_U_HALF) | (state.numel() == 0 ? CASTLE_FLAG_RECOMPUTE_STATE : 0);   // U_HALF describes the forward's U output only
}
int64_t bwd_workspace_bytes(const Shape& s, int64_t flags, const Tensor& state) {
  return check(castle_bwd_workspace_bytes(s.B, s.H, s.L, s.d, s.dtype, bwd_flags(flags, state)), "castle_bwd_workspace_bytes");
}

// grads: dqc, dkc, dvc, dqu, dku, dvu.  The backward kernels take the operands from the copies in the forward workspace.
void run_bwd(const castle_view4 (&six)[6], const castle_view4& out, const castle_view4& dout, const Shape& s, double scale, int64_t flags,
             const castle_view4 (&grads)[6], const Tensor& ws, const Tensor& state, const Tensor& prepared = Tensor()) {
  // prepared: a backward workspace that holds the partial maxima of |dout| already
  int fl = bwd_flags(flags, state);
  const int64_t nbytes = bwd_workspace_bytes(s, flags, state);
  Tensor bws = prepared.defined() ? prepared : bytes(nbytes, ws);
  if (prepared.defined()) fl |= CASTLE_FLAG_AMAX_READY;
  check(castle_bwd(&six[0], &six[1], &six[2], &six[3], &six[4], &six[5], &out, &dout, s.B, s.H, s.L, s.d, s.dtype, (float)scale, fl,
                   &grads[0], &grads[1], &grads[2], &grads[3], &grads[4], &grads[5], ws.data_ptr(), ws.numel(),
                   state.numel() ? state.data_ptr() : nullptr, state.numel(), bws.data_ptr(), nbytes, stream_of(ws)),
        "castle_bwd");
}

void require_gpu(const Tensor& t, const char* what) {
  TORCH_CHECK(t.is_cuda(), what, ": the HIP kernels need tensors on the GPU (got ", t.device(), ")");
}

// ---- the operator on six (B, H, L, d) tensors ------------------------------------------------------------------
Shape shape_of(const Tensor& q) { return {(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)q.size(3), dtype_code(q)}; }

std::tuple<Tensor, Tensor, Tensor, Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qu, const Tensor& ku,
                                                     const Tensor& vu, double scale, bool want_U, int64_t flags, bool keep_state) {
  require_gpu(q, "castle_attention_hip");
  check_dims(q.size(3), q);
  const Shape s = shape_of(q);
  const c10::DeviceGuard guard(q.device());
  const Tensor ops[6] = {readable(q), readable(k), readable(v), readable(qu), readable(ku), readable(vu)};
  castle_view4 six[6];
  for (int i = 0; i < 6; ++i) six[i] = view4(ops[i]);
  const int64_t B = s.B, H = s.H, L = s.L, d = s.d;
  Tensor out = at::empty({B, L, H, d}, q.options()).permute({0, 2, 1, 3});
  Tensor U = want_U ? at::empty({B, H, L, d}, q.options()) : at::empty({0}, q.options());
  auto [ws, state] = run_fwd(six, s, scale, flags, view4(out), want_U ? view4(U) : castle_view4{nullptr, 0, 0, 0}, keep_state, q);
  return {out, U, ws, state};
}

Tensor attention_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qu, const Tensor& ku, const Tensor& vu,
                     const Tensor& out, const Tensor& dout, const Tensor& ws, const Tensor& state, double scale, int64_t flags) {
  const Shape s = shape_of(q);
  const c10::DeviceGuard guard(q.device());
  const Tensor ops[8] = {readable(q), readable(k), readable(v), readable(qu), readable(ku), readable(vu), readable(out), readable(dout)};
  castle_view4 six[6], grads[6];
  for (int i = 0; i < 6; ++i) six[i] = view4(ops[i]);
  const int64_t B = s.B, H = s.H, L = s.L, d = s.d;
  Tensor packed = at::empty({6, B, H, L, d}, out.options());
  for (int i = 0; i < 6; ++i)
    grads[i] = {static_cast<char*>(packed.data_ptr()) + i * B * H * L * d * packed.element_size(), H * L * d, L * d, d};
  run_bwd(six, view4(ops[6]), view4(ops[7]), s, scale, flags, grads, ws, state);
  return packed;
}

// ---- the operator on the fused projection (B, L, 6 H d), order qu, ku, vu, qc, kc, vc --------------------------
Shape packed_shape(const Tensor& proj, int64_t heads) {
  return {(int)proj.size(0), (int)heads, (int)proj.size(1), (int)(proj.size(2) / (6 * heads)), dtype_code(proj)};
}
void six_of_packed(const Tensor& p, const Shape& s, castle_view4 (&six)[6]) {
  for (int i = 0; i < 3; ++i) {
    six[i] = packed_view(p, s, 6, 3 + i);
    six[3 + i] = packed_view(p, s, 6, i);
  }
}

std::tuple<Tensor, Tensor, Tensor, Tensor> run_packed(const Tensor& proj, int64_t heads, double scale, bool want_U,
                                                            int64_t row_capacity, int64_t flags, bool keep_state, const Tensor& prepared,
                                                            const Tensor& U_buffer = Tensor()) {
  // The lookahead keys come back as the first L rows of a (B, H, row_capacity, d) buffer, `U_buffer` if there is one, so that a
  // caller can hand over the U buffer of a decode cache without copying (row_capacity >= L).
  require_gpu(proj, "castle_attention_packed");
  const Shape s = packed_shape(proj, heads);
  check_dims(s.d, proj);
  const c10::DeviceGuard guard(proj.device());
  const Tensor p = packed_readable(proj);
  castle_view4 six[6];
  six_of_packed(p, s, six);
  const int64_t B = s.B, H = s.H, L = s.L, d = s.d, cap = std::max(row_capacity, L);
  Tensor merged = at::empty({B, L, H * d}, proj.options());
  Tensor U = U_buffer.defined() ? U_buffer : want_U ? at::empty({B, H, cap, d}, proj.options()) : at::empty({0}, proj.options());
  auto [ws, state] = run_fwd(six, s, scale, flags, packed_view(merged, s, 1, 0),
                             want_U ? view4(U) : castle_view4{nullptr, 0, 0, 0}, keep_state, proj, prepared);
  return {merged, U, ws, state};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> attention_packed(const Tensor& proj, int64_t heads, double scale, bool want_U,
                                                            int64_t row_capacity, int64_t flags, bool keep_state) {
  return run_packed(proj, heads, scale, want_U, row_capacity, flags, keep_state, Tensor());
}

Tensor attention_packed_bwd(const Tensor& proj, const Tensor& merged, const Tensor& dmerged, const Tensor& ws, const Tensor& state,
                            int64_t heads, double scale, int64_t flags) {
  const Shape s = packed_shape(proj, heads);
  const c10::DeviceGuard guard(proj.device());
  const Tensor p = packed_readable(proj), dm = packed_readable(dmerged);
  Tensor dproj = at::empty(proj.sizes(), proj.options());
  castle_view4 six[6], grads[6];
  six_of_packed(p, s, six);
  six_of_packed(dproj, s, grads);
  run_bwd(six, packed_view(merged, s, 1, 0), packed_view(dm, s, 1, 0), s, scale, flags, grads, ws, state);
  return dproj;
}

// ---- autograd ----------------------------------------------------------------------------------------------------
// U, the workspace and the state carry no gradient (lookahead_keys_attention_triton.py:513-515 for U), and
// autograd does not materialise zeros for them (a fill of hundreds of MB per backward pass).  The formulas call
// the backward operators through the dispatcher, so that they trace like any other operator.  A graph that was traced without
// gradients carries CASTLE_FLAG_FORWARD_ONLY in its arguments: where it runs with gradients, the flag is dropped.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Whether a call records a graph.
bool wants_graph(std::initializer_list<Tensor> ts) {
  bool graph = false;
  for (const Tensor& t : ts) {
    if (!t.defined()) continue;
    no_tangent(t);
    graph = graph || t.requires_grad();
  }
  return graph && at::GradMode::is_enabled();
}

// The gradients have no derivatives of their own.  Where a graph of the backward pass is recorded (create_graph) they hang on a
// node that raises when somebody differentiates them: as constants, a penalty on them would add nothing, without a word.
variable_list no_second_derivatives(const variable_list& grads) {
  variable_list alias;
  alias.reserve(grads.size());
  for (const Tensor& t : grads) alias.push_back(t.defined() ? t.detach().set_requires_grad(true) : t);
  const auto raises = std::make_shared<torch::autograd::DelayedError>(
      "trying to differentiate twice through the CASTLE kernels: their gradients have no derivatives (Castle(use_triton=False) is "
      "differentiable any number of times)", (int64_t)grads.size());
  return (*raises)(std::move(alias));
}
template <typename F> variable_list once_differentiable(F&& gradients) {
  variable_list grads;
  {
    const at::NoGradGuard no_grad;
    grads = gradients();
  }
  if (at::GradMode::is_enabled()) return no_second_derivatives(grads);
  return grads;
}

template <typename F> auto op_handle(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}

struct AttentionFn : torch::autograd::Function<AttentionFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qu,
                               const Tensor& ku, const Tensor& vu, double scale, bool want_U, int64_t flags, bool keep_state) {
    static const auto op = op_handle<decltype(attention)>("castle_hip::attention");
    flags &= ~CASTLE_FLAG_FORWARD_ONLY;
    const at::AutoDispatchBelowADInplaceOrView below;
    auto [out, U, ws, state] = op.call(q, k, v, qu, ku, vu, scale, want_U, flags, keep_state);
    ctx->save_for_backward({q, k, v, qu, ku, vu, out, ws, state});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = flags;
    ctx->mark_non_differentiable({U, ws, state});
    ctx->set_materialize_grads(false);
    return {out, U, ws, state};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    static const auto op = op_handle<decltype(attention_bwd)>("castle_hip::attention_bwd");
    const auto s = ctx->get_saved_variables();
    const Tensor dout = g[0].defined() ? g[0] : at::zeros_like(s[6]);
    const auto d = op.call(s[0], s[1], s[2], s[3], s[4], s[5], s[6], dout, s[7], s[8], ctx->saved_data["scale"].toDouble(),
                           ctx->saved_data["flags"].toInt()).unbind(0);
    return {d[0], d[1], d[2], d[3], d[4], d[5], Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor attention_bwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qu, const Tensor& ku, const Tensor& vu,
                              const Tensor& out, const Tensor& dout, const Tensor& ws, const Tensor& state, double scale, int64_t flags) {
  static const auto op = op_handle<decltype(attention_bwd)>("castle_hip::attention_bwd");
  const bool graph = wants_graph({q, k, v, qu, ku, vu, out, dout});
  const at::AutoDispatchBelowADInplaceOrView below;
  const Tensor d = op.call(q, k, v, qu, ku, vu, out, dout, ws, state, scale, flags);
  return graph ? no_second_derivatives({d})[0] : d;
}

std::tuple<Tensor, Tensor, Tensor, Tensor> attention_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qu,
                                                              const Tensor& ku, const Tensor& vu, double scale, bool want_U,
                                                              int64_t flags, bool keep_state) {
  if (!wants_graph({q, k, v, qu, ku, vu})) {
    static const auto op = op_handle<decltype(attention)>("castle_hip::attention");
    const at::AutoDispatchBelowADInplaceOrView below;
    return op.call(q, k, v, qu, ku, vu, scale, want_U, flags, keep_state);
  }
  auto r = AttentionFn::apply(q, k, v, qu, ku, vu, scale, want_U, flags, keep_state);
  return {r[0], r[1], r[2], r[3]};
}

struct AttentionPackedFn : torch::autograd::Function<AttentionPackedFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& proj, int64_t heads, double scale, bool want_U, int64_t row_capacity,
                               int64_t flags, bool keep_state) {
    static const auto op = op_handle<decltype(attention_packed)>("castle_hip::attention_packed");
    flags &= ~CASTLE_FLAG_FORWARD_ONLY;
    const at::AutoDispatchBelowADInplaceOrView below;
    auto [merged, U, ws, state] = op.call(proj, heads, scale, want_U, row_capacity, flags, keep_state);
    ctx->save_for_backward({proj, merged, ws, state});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = flags;
    ctx->mark_non_differentiable({U, ws, state});
    ctx->set_materialize_grads(false);
    return {merged, U, ws, state};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    static const auto op = op_handle<decltype(attention_packed_bwd)>("castle_hip::attention_packed_bwd");
    const auto s = ctx->get_saved_variables();
    const Tensor dm = g[0].defined() ? g[0] : at::zeros_like(s[1]);
    Tensor dproj = op.call(s[0], s[1], dm, s[2], s[3], ctx->saved_data["heads"].toInt(), ctx->saved_data["scale"].toDouble(),
                           ctx->saved_data["flags"].toInt());
    return {dproj, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor attention_packed_bwd_autograd(const Tensor& proj, const Tensor& merged, const Tensor& dmerged, const Tensor& ws, const Tensor& state,
                                     int64_t heads, double scale, int64_t flags) {
  static const auto op = op_handle<decltype(attention_packed_bwd)>("castle_hip::attention_packed_bwd");
  const bool graph = wants_graph({proj, merged, dmerged});
  const at::AutoDispatchBelowADInplaceOrView below;
  const Tensor d = op.call(proj, merged, dmerged, ws, state, heads, scale, flags);
  return graph ? no_second_derivatives({d})[0] : d;
}

std::tuple<Tensor, Tensor, Tensor, Tensor> attention_packed_autograd(const Tensor& proj, int64_t heads, double scale, bool want_U,
                                                                     int64_t row_capacity, int64_t flags, bool keep_state) {
  if (!wants_graph({proj})) {
    static const auto op = op_handle<decltype(attention_packed)>("castle_hip::attention_packed");
    const at::AutoDispatchBelowADInplaceOrView below;
    return op.call(proj, heads, scale, want_U, row_capacity, flags, keep_state);
  }
  auto r = AttentionPackedFn::apply(proj, heads, scale, want_U, row_capacity, flags, keep_state);
  return {r[0], r[1], r[2], r[3]};
}

// ---- rows between the products ---------------------------------------------------------------------------------
// F.rms_norm on the GPU without an eps takes the epsilon of its 32-bit sums, whatever the type of the rows
double norm_eps(std::optional<double> eps) { return eps.value_or(1.1920928955078125e-07); }

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
Tensor row_major(const Tensor& t) { return t.is_contiguous() && aligned16(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

struct Normed {
  Tensor sum, h, rstd;   // sum: x, or x + delta; rstd is only there for a backward pass
};
// RMS norm of (R, D) rows, of x or of x + delta; without a weight h is the sum itself.  Rows longer than the kernels
// hold in registers take the library's norm.
Normed norm_rows(const Tensor& x_, const Tensor& delta_, const Tensor& w_, std::optional<double> eps, bool want_rstd) {
  if (!w_.defined()) {
    const Tensor sum = delta_.defined() ? x_ + delta_ : x_;
    return {sum, sum, Tensor()};
  }
  const int64_t R = x_.size(0), D = x_.size(1);
  TORCH_CHECK_VALUE(w_.numel() == D && w_.device() == x_.device() && w_.scalar_type() == x_.scalar_type() &&
                        (!delta_.defined() || (delta_.sizes() == x_.sizes() && delta_.device() == x_.device() && delta_.scalar_type() == x_.scalar_type())),
                    "the norm's weight or the summand does not belong to these rows");
  if (castle_rms_norm_bwd_workspace_bytes(R, (int)D, dtype_code(x_)) < 0) {
    const Tensor sum = delta_.defined() ? x_ + delta_ : x_;
    auto [h, rstd] = at::_fused_rms_norm(sum, {D}, w_, eps);
    return {sum, h, rstd};
  }
  const Tensor x = row_major(x_), w = row_major(w_), delta = delta_.defined() ? row_major(delta_) : Tensor();
  Tensor sum = delta.defined() ? at::empty_like(x) : x, h = at::empty_like(x), rstd = want_rstd ? at::empty({R}, x.options().dtype(at::kFloat)) : Tensor();
  check(castle_rms_norm(x.data_ptr(), delta.defined() ? delta.data_ptr() : nullptr, w.data_ptr(), delta.defined() ? sum.data_ptr() : nullptr, h.data_ptr(),
                        want_rstd ? static_cast<float*>(rstd.data_ptr()) : nullptr, R, (int)D, (float)norm_eps(eps), dtype_code(x), stream_of(x)),
        "castle_rms_norm");
  return {sum, h, rstd};
}
// dh -> (dres + gradient of the rows, gradient of the weight); rstd as norm_rows left it
constexpr int64_t kSumsBytes = 4 << 20;
// Sums of partial weight gradients that wait for the end of a backward pass, for one launch instead of one each (4 us each for a MB or two).
struct Sums {
  castle_sum sum[CASTLE_MAX_SUMS];
  Tensor keep[2 * CASTLE_MAX_SUMS];   // what they read and write
  int count = 0;
  // what is larger is not in a cache any more when it is read (50 MB behind the input gradient of 16384 rows: 1 to 2 us lost, not won)
  bool takes(int64_t parts, int64_t n) const { return parts * n * 4 <= kSumsBytes && count < CASTLE_MAX_SUMS; }
  void add(const castle_sum& s, const Tensor& part, const Tensor& out) {
    if (s.parts == 0) return;
    sum[count] = s;
    keep[2 * count] = part;
    keep[2 * count++ + 1] = out;
  }
  void flush() {
    if (count == 0) return;
    check(castle_sums(sum, count, dtype_code(keep[1]), stream_of(keep[1])), "castle_sums");
    count = 0;
    for (Tensor& t : keep) t = Tensor();
  }
};

std::tuple<Tensor, Tensor> norm_rows_bwd(const Tensor& dh_, const Tensor& x_, const Tensor& rstd, const Tensor& w_, const Tensor& dres_, bool need_x,
                                         bool need_w, Sums* sums = nullptr) {
  if (!w_.defined()) return {dres_.defined() ? dres_ + dh_ : dh_, Tensor()};
  const int64_t R = x_.size(0), D = x_.size(1);
  if (rstd.dim() != 1) {
    auto [dx, dw] = at::_fused_rms_norm_backward(dh_, x_, {D}, rstd, w_, {need_x, need_w});
    return {need_x && dres_.defined() ? dres_ + dx : dx, dw};
  }
  const Tensor x = row_major(x_), dh = row_major(dh_), w = row_major(w_), dres = need_x && dres_.defined() ? row_major(dres_) : Tensor();
  const int64_t nbytes = need_w ? castle_rms_norm_bwd_workspace_bytes(R, (int)D, dtype_code(x)) : 0;
  Tensor dx = need_x ? at::empty_like(x) : Tensor(), dw = need_w ? at::empty_like(w) : Tensor(), ws = need_w ? bytes(nbytes, x) : Tensor();
  if (sums != nullptr && need_w && sums->takes(1, nbytes / 4)) {
    castle_sum sum;
    check(castle_rms_norm_bwd_parts(dh.data_ptr(), x.data_ptr(), w.data_ptr(), static_cast<const float*>(rstd.data_ptr()), dres.defined() ? dres.data_ptr() : nullptr,
                                    need_x ? dx.data_ptr() : nullptr, dw.data_ptr(), &sum, R, (int)D, dtype_code(x), ws.data_ptr(), nbytes, stream_of(x)),
          "castle_rms_norm_bwd_parts");
    sums->add(sum, ws, dw);
    return {dx, dw};
  }
  check(castle_rms_norm_bwd(dh.data_ptr(), x.data_ptr(), w.data_ptr(), static_cast<const float*>(rstd.data_ptr()), dres.defined() ? dres.data_ptr() : nullptr,
                            need_x ? dx.data_ptr() : nullptr, need_w ? dw.data_ptr() : nullptr, R, (int)D, dtype_code(x),
                            need_w ? ws.data_ptr() : nullptr, nbytes, stream_of(x)),
        "castle_rms_norm_bwd");
  return {dx, dw};
}

// The norm as a registered operator, for callers that are traced: what they record is what an untraced layer runs.
std::tuple<Tensor, Tensor> rms_norm_op(const Tensor& x, const Tensor& weight, std::optional<double> eps) {
  const c10::DeviceGuard guard(x.device());
  const Normed n = norm_rows(x.reshape({-1, x.size(-1)}), Tensor(), weight, eps, true);
  return {n.h.view(x.sizes()), n.rstd};
}
// (a gradient that is not asked for, of a frozen weight for instance, comes back empty)
std::tuple<Tensor, Tensor> rms_norm_bwd_op(const Tensor& dh, const Tensor& x, const Tensor& rstd, const Tensor& weight, bool need_x, bool need_w) {
  const c10::DeviceGuard guard(x.device());
  const int64_t D = x.size(-1);
  if (!need_x && !need_w) return {at::empty({0}, x.options()), at::empty({0}, weight.options())};
  auto [dx, dw] = norm_rows_bwd(dh.reshape({-1, D}), x.reshape({-1, D}), rstd, weight, Tensor(), need_x, need_w);
  return {need_x ? dx.view(x.sizes()) : at::empty({0}, x.options()), need_w ? dw : at::empty({0}, weight.options())};
}
struct RmsNormFn : torch::autograd::Function<RmsNormFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, std::optional<double> eps) {
    static const auto op = op_handle<decltype(rms_norm_op)>("castle_hip::rms_norm");
    const at::AutoDispatchBelowADInplaceOrView below;
    auto [h, rstd] = op.call(x, weight, eps);
    ctx->save_for_backward({x, rstd, weight});
    ctx->mark_non_differentiable({rstd});
    ctx->set_materialize_grads(false);
    return {h, rstd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    static const auto op = op_handle<decltype(rms_norm_bwd_op)>("castle_hip::rms_norm_bwd");
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
    auto [dx, dw] = op.call(g[0], s[0], s[1], s[2], need_x, need_w);
    return {need_x ? dx : Tensor(), need_w ? dw : Tensor(), Tensor()};
  }
};
std::tuple<Tensor, Tensor> rms_norm_bwd_autograd(const Tensor& dh, const Tensor& x, const Tensor& rstd, const Tensor& weight, bool need_x, bool need_w) {
  static const auto op = op_handle<decltype(rms_norm_bwd_op)>("castle_hip::rms_norm_bwd");
  const bool graph = wants_graph({dh, x, weight});
  const at::AutoDispatchBelowADInplaceOrView below;
  const auto [dx, dw] = op.call(dh, x, rstd, weight, need_x, need_w);
  if (!graph) return {dx, dw};
  const auto r = no_second_derivatives({dx, dw});
  return {r[0], r[1]};
}
std::tuple<Tensor, Tensor> rms_norm_autograd(const Tensor& x, const Tensor& weight, std::optional<double> eps) {
  if (!wants_graph({x, weight})) {
    static const auto op = op_handle<decltype(rms_norm_op)>("castle_hip::rms_norm");
    const at::AutoDispatchBelowADInplaceOrView below;
    return op.call(x, weight, eps);
  }
  auto r = RmsNormFn::apply(x, weight, eps);
  return {r[0], r[1]};
}

// a (M, K), or (K, M) with a_t; b (N, K), or (K, N) with b_t -> (M, N); rows contiguous up to a leading dimension (not
// repeated or overlapping ones), the last element within reach of the kernel's 32-bit offsets
bool product_rows(const Tensor& t) {
  return t.dim() == 2 && t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % (16 / t.element_size()) == 0 && t.size(1) % (16 / t.element_size()) == 0 && aligned16(t) &&
         castle_gemm_operand_ok(t.size(0), t.stride(0));
}
Tensor product(const Tensor& a, bool a_t, const Tensor& b, bool b_t, int64_t epilogue, const std::optional<Tensor>& aux, const castle_amax* amax = nullptr) {
  const c10::DeviceGuard guard(a.device());
  TORCH_CHECK_VALUE(product_rows(a) && product_rows(b), "product: unexpected operands");
  const int64_t M = a.size(a_t ? 1 : 0), K = a.size(a_t ? 0 : 1), N = b.size(b_t ? 1 : 0);
  TORCH_CHECK_VALUE(b.size(b_t ? 0 : 1) == K && b.device() == a.device() && b.scalar_type() == a.scalar_type(), "product: operands do not match");
  const int dtype = dtype_code(a);
  const int64_t nbytes = check(castle_gemm_workspace_bytes((int)M, (int)N, (int)K, dtype, (int)epilogue), "castle_gemm_workspace_bytes");
  Tensor c = at::empty({M, N}, a.options()), ws = nbytes ? bytes(nbytes, a) : Tensor();
  TORCH_CHECK_VALUE(!aux || (aux->is_contiguous() && aux->sizes() == c.sizes() && aux->scalar_type() == c.scalar_type() && aux->device() == c.device()),
                    "product: unexpected second tensor");
  check(castle_gemm(a.data_ptr(), a.stride(0), a_t, b.data_ptr(), b.stride(0), b_t, c.data_ptr(), N, (int)M, (int)N, (int)K, dtype, (int)epilogue,
                    aux ? aux->data_ptr() : nullptr, amax, nbytes ? ws.data_ptr() : nullptr, nbytes, stream_of(a)),
        "castle_gemm");
  return c;
}

// ---- projections -----------------------------------------------------------------------------------------------
// Own products where a call is short: the library's costs 18 us of host time, one here 4.  On the GPU they are level or
// ahead up to the sizes below (us, own / library: input gradient of 1000 rows x 3072 x 512 15 / 16, 4096 x 3072 x 512 31 / 31, 8192 x 3072 x
// 512 44 / 39; weight gradient of 3000 rows, 1536 x 256, 14 / 27, of 4096, 3072 x 512, 31 / 41; forward of 4096 rows 1024 -> 3072 31 / 30).
// Contractions of up to 512 in whole steps of 64: ahead at every size measured up to 309 GFLOP (the line lies between that and 206), since a tile's start
// and end weigh more there than its steps, and the store takes gelu and the maxima along (forward / input gradient, 16384 rows 64 -> 3072 24 / 29 and
// 24 / 30, 128 -> 3072 30 / 32 and 31 / 35, 256 -> 3072 38 / 43 and 38 / 45, 512 -> 3072 59 / 62 and 59 / 67, 512 -> 512 14 / 20 and 14 / 20; 65536 rows 64 -> 3072 81 /
// 100 and 82 / 105, 128 -> 3072 103 / 126 and 105 / 129, 512 -> 3072 227 / 240 and 228 / 253; 98304 rows 354 / 359 and 361 / 379, 131072 rows 478 / 473 and 484 /
// 500).  Longer ones are level at 16384 rows (forward 576 -> 3072 64 / 59, 640 68 / 64, 768 76 / 72).
// In fp32 they are ahead at nearly every size, up to the largest that was timed, 825 GFLOP (us, own / library: 16384 rows 2048 -> 12288 forward 4950 / 5530, input
// gradient 4840 / 5350, weight gradient 4820 / 5360; 256 rows 512 -> 3072 11 / 13, 15 / 13 and 11 / 17).
bool own_product(const Tensor& a, const Tensor& b, int64_t rows, int64_t n, int64_t k, double most_16) {
  return (a.scalar_type() == at::kFloat || 2.0 * rows * n * k <= most_16) && n % 8 == 0 && k % 8 == 0 && product_rows(a) && product_rows(b);
}
bool own_contraction(int64_t k) { return k <= 512 && k % 64 == 0; }   // (others have no tiles of 256 rows)
double own_forward(int64_t k) { return own_contraction(k) ? 260e9 : 14e9; }
double own_input_grad(int64_t k) { return own_contraction(k) ? 260e9 : 4e9; }
constexpr double kOwnWeightGrad = 40e9;
constexpr double kOwnGeluSlope = 40e9;   // the pass it saves over the hidden rows outweighs a slower product: 16384 x 512 x 2048 73 / 91

// The attention kernels behind a product begin with the largest element of some of its columns (vu of a fused projection, all
// of the gradient of the merged heads): an own product leaves the partial maxima where they look for them, in the
// workspace that is then handed on (`prepared`; undefined when there are none: fp32, the library's product, a split contraction).
struct Maxima {
  Tensor prepared;
  castle_amax where;
  const castle_amax* get() const { return prepared.defined() ? &where : nullptr; }
};
Maxima maxima(const Tensor& like, int64_t rows, int64_t n, int64_t k, int64_t column, int64_t columns, int64_t nbytes, bool status) {
  Maxima m;
  if (like.scalar_type() == at::kFloat || !castle_gemm_amax_ok((int)rows, (int)n, (int)k, dtype_code(like), (int)column, (int)columns)) return m;
  m.prepared = bytes(nbytes, like);
  char* p = static_cast<char*>(m.prepared.data_ptr());
  m.where = {reinterpret_cast<float*>(p + CASTLE_AMAX_OFFSET), status ? reinterpret_cast<int*>(p) : nullptr, (int32_t)column, (int32_t)columns};
  return m;
}

Tensor project(const Tensor& x, const Tensor& w) {   // (R, K), (N, K) -> (R, N)
  if (own_product(x, w, x.size(0), w.size(0), x.size(1), own_forward(x.size(1)))) return product(x, false, w, false, CASTLE_GEMM_PLAIN, std::nullopt);
  return at::mm(x, w.t());
}
// the fused projection, with the maxima of its vu part
Maxima packed_maxima(const Tensor& x, const Tensor& w, const Shape& s) {
  const int64_t part = (int64_t)s.H * s.d;
  return maxima(x, x.size(0), w.size(0), x.size(1), 2 * part, part, check(castle_fwd_workspace_bytes(s.B, s.H, s.L, s.d, s.dtype), "castle_fwd_workspace_bytes"), true);
}
Tensor project_packed(const Tensor& x, const Tensor& w, const Shape& s, Tensor& prepared) {
  if (!own_product(x, w, x.size(0), w.size(0), x.size(1), own_forward(x.size(1)))) return at::mm(x, w.t());
  const Maxima m = packed_maxima(x, w, s);
  prepared = m.prepared;
  return product(x, false, w, false, CASTLE_GEMM_PLAIN, std::nullopt, m.get());
}
// Few rows are normalised inside the product that reads them: a launch less (a layer over one sequence of 96 rows 30.9 -> 25.8 us).
bool norm_in_product(const Tensor& x, const Tensor& norm_w, const Tensor& w) {
  const int64_t R = x.size(0), D = x.size(1);
  return norm_w.defined() && norm_w.numel() == D && norm_w.is_contiguous() && norm_w.device() == x.device() && norm_w.scalar_type() == x.scalar_type() &&
         x.is_contiguous() && w.size(1) == D && w.device() == x.device() && w.scalar_type() == x.scalar_type() && castle_rms_norm_bwd_workspace_bytes(R, (int)D, dtype_code(x)) >= 0 &&
         own_product(x, w, R, w.size(0), D, own_forward(D)) && castle_gemm_norm_ok((int)R, (int)w.size(0), (int)D, dtype_code(x));
}
// the same behind the norm; n.h and n.rstd are left where something will read them
Tensor project_packed_of_norm(const Tensor& x, const Tensor& norm_w, std::optional<double> eps, const Tensor& w, const Shape& s, bool keep, Normed& n, Tensor& prepared) {
  const Maxima m = packed_maxima(x, w, s);
  prepared = m.prepared;
  const int64_t R = x.size(0), D = x.size(1), N = w.size(0);
  n = {x, keep ? at::empty_like(x) : Tensor(), keep ? at::empty({R}, x.options().dtype(at::kFloat)) : Tensor()};
  const castle_gemm_norm norm = {norm_w.data_ptr(), (float)norm_eps(eps), keep ? n.h.data_ptr() : nullptr, keep ? static_cast<float*>(n.rstd.data_ptr()) : nullptr};
  Tensor c = at::empty({R, N}, x.options());
  check(castle_gemm_of_norm(x.data_ptr(), D, &norm, w.data_ptr(), w.stride(0), c.data_ptr(), N, (int)R, (int)N, (int)D, dtype_code(x), m.get(), stream_of(x)),
        "castle_gemm_of_norm");
  return c;
}
Tensor input_grad(const Tensor& dy, const Tensor& w) {   // (R, N), (N, K) -> (R, K)
  if (own_product(dy, w, dy.size(0), w.size(0), w.size(1), own_input_grad(w.size(0)))) return product(dy, false, w, true, CASTLE_GEMM_PLAIN, std::nullopt);
  return at::mm(dy, w);
}

// The weight gradient of a projection over many rows, dW = dY^T x, is a product with a small output
// (out_features x in_features) and a long contraction (the rows): the GEMM the library picks leaves most of
// the GPU idle there.  From kSplitWgradMinRows rows on it is formed as partial products over row ranges (one batched GEMM
// with fp32 partial results, then their sum; same rounding), as many as make about 256 tiles of 256 x 256: 16384 rows,
// us as one product / with 2, 4, 8 ranges and their sum: 3072 x 512 123 / 80, 64, 63; 2048 x 2048 153 / 137, 139, 161;
// 6144 x 1024 214 / 187, 200, 231; 12288 x 2048 890 / 931, 884, 1000.
// Up to 32 GFLOP the framework's own product, which splits the rows by what fills the CUs, is ahead of that: over 2500 of 8192 ... 65536 rows, widths of 64 ... 6144
// in bf16, partial products and their sum take 1.18 times as long below 1 GFLOP, 1.39 at 1 to 2, 1.55 at 2 to 8, 1.41 at 8 to 16, 1.28 at 16 to 32 (less than 0.97
// times in 1 of 100 above 1 GFLOP), 1.16 at 32 to 40 with 1 of 13 behind, 1.00 from 64 on.  24000 rows 256 x 256 27.5 / 19.4, 16384 rows 768 x 128 25.1 / 18.8.  Rows that do not split
// evenly leave the library one product: behind up to what was timed, 130 GFLOP (2.0 times at 40 to 64, 1.6 beyond).
constexpr int64_t kSplitWgradMinRows = 8192;
double own_weight_grad(const Tensor& x, int64_t rows, int64_t parts) {
  return x.scalar_type() == at::kFloat || rows < kSplitWgradMinRows ? kOwnWeightGrad : rows % parts == 0 ? 32e9 : 130e9;
}
int64_t wgrad_parts(int64_t N, int64_t K) {
  const int64_t tiles = ((N + 255) / 256) * ((K + 255) / 256);
  return tiles >= 192 ? 1 : tiles >= 96 ? 2 : tiles >= 48 ? 4 : 8;
}

Tensor weight_grad(const Tensor& dy, const Tensor& x, Sums* sums = nullptr) {   // (R, N), (R, K) -> (N, K)
  const int64_t rows = x.size(0), N = dy.size(1), K = x.size(1);
  const int64_t parts = wgrad_parts(N, K);
  if (own_product(dy, x, rows, N, K, own_weight_grad(x, rows, parts))) return product(dy, true, x, true, CASTLE_GEMM_PLAIN, std::nullopt);
  if (x.scalar_type() != at::kFloat && rows >= kSplitWgradMinRows && rows % parts == 0 && N * K % 8 == 0) {
    if (parts == 1) return at::mm(dy.t(), x);
    const int64_t r = rows / parts;
    const Tensor a = dy.contiguous().view({parts, r, N}).transpose(1, 2);
    const Tensor part = at::bmm(a, x.contiguous().view({parts, r, K}), at::kFloat).contiguous();
    Tensor dw = at::empty({N, K}, x.options());
    if (sums != nullptr && sums->takes(parts, N * K)) {
      sums->add({static_cast<const float*>(part.data_ptr()), N * K, dw.data_ptr(), (int32_t)parts, 0}, part, dw);
      return dw;
    }
    check(castle_sum_parts(static_cast<const float*>(part.data_ptr()), (int)parts, N * K, dw.data_ptr(), dtype_code(x), stream_of(x)),
          "castle_sum_parts");
    return dw;
  }
  return at::mm(dy.t(), x);
}

constexpr double kOwnLongGrads = 8e9;   // 16-bit: from kSplitWgradMinRows rows on both in one launch take 1/1.32 of two up to here, more of some from 12 GFLOP on
// Both gradients of a projection, in one launch where that is ahead (false: they are left to the functions above).  aux: dx is multiplied by the slope of gelu at
// it; nbytes >= 0: the maxima of |dx| go to a workspace of that size, `prepared` (16-bit types).
bool own_projection_grads(const Tensor& dy, const Tensor& x, const Tensor& w, const Tensor& aux, int64_t nbytes, Tensor& dw, Tensor& dx, Tensor& prepared, Sums* sums = nullptr) {
  const int64_t R = dy.size(0), N = dy.size(1), K = w.size(1);
  const bool full = dy.scalar_type() == at::kFloat, with_amax = !full && nbytes >= 0;
  if (x.dim() != 2 || x.size(0) != R || x.size(1) != K || w.size(0) != N || x.scalar_type() != dy.scalar_type() || w.scalar_type() != dy.scalar_type() || x.device() != dy.device() ||
      w.device() != dy.device() || !own_product(dy, x, R, N, K, !full && R >= kSplitWgradMinRows ? kOwnLongGrads : kOwnWeightGrad) ||
      !own_product(dy, w, R, K, N, aux.defined() ? kOwnGeluSlope : own_input_grad(N)))
    return false;
  if (aux.defined() && !(aux.is_contiguous() && aux.dim() == 2 && aux.size(0) == R && aux.size(1) == K && aux.scalar_type() == dy.scalar_type() && aux.device() == dy.device() && aligned16(aux)))
    return false;
  const int dtype = dtype_code(dy), epilogue = aux.defined() ? CASTLE_GEMM_GELU_SLOPE : CASTLE_GEMM_PLAIN;
  const int64_t need = castle_projection_grads_workspace_bytes((int)R, (int)N, (int)K, dtype, epilogue, with_amax);
  if (need < 0) return false;
  castle_amax where;
  if (with_amax) {
    prepared = bytes(nbytes, dy);
    where = {reinterpret_cast<float*>(static_cast<char*>(prepared.data_ptr()) + CASTLE_AMAX_OFFSET), nullptr, 0, (int32_t)K};
  }
  const Tensor ws = need ? bytes(need, dy) : Tensor();
  dw = at::empty({N, K}, dy.options());
  dx = at::empty({R, K}, dy.options());
  castle_sum sum = {};
  const bool later = sums != nullptr && sums->takes(1, need / 4);
  check(castle_projection_grads(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), dw.data_ptr(), dx.data_ptr(), (int)R, (int)N, (int)K, dtype,
                                epilogue, aux.defined() ? aux.data_ptr() : nullptr, with_amax ? &where : nullptr, later ? &sum : nullptr, need ? ws.data_ptr() : nullptr, need, stream_of(dy)),
        "castle_projection_grads");
  if (later) sums->add(sum, ws, dw);
  return true;
}

// A projection as a registered operator, for callers that are traced.
Tensor linear_op(const Tensor& x, const Tensor& weight) {
  const c10::DeviceGuard guard(x.device());
  std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = weight.size(0);
  return project(x.reshape({-1, x.size(-1)}), weight).view(shape);
}
std::tuple<Tensor, Tensor> linear_bwd_op(const Tensor& dy_, const Tensor& x, const Tensor& weight, bool need_x, bool need_w) {
  const c10::DeviceGuard guard(x.device());
  const Tensor dy = dy_.reshape({-1, weight.size(0)});
  Tensor dw, dx, none;
  if (need_x && need_w && own_projection_grads(dy, x.reshape({-1, x.size(-1)}), weight, Tensor(), -1, dw, dx, none)) return {dx.view(x.sizes()), dw};
  return {need_x ? input_grad(dy, weight).view(x.sizes()) : at::empty({0}, x.options()),
          need_w ? weight_grad(dy, x.reshape({-1, x.size(-1)})) : at::empty({0}, weight.options())};
}
struct LinearFn : torch::autograd::Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight) {
    static const auto op = op_handle<decltype(linear_op)>("castle_hip::linear");
    const at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({x, weight});
    return op.call(x, weight);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    static const auto op = op_handle<decltype(linear_bwd_op)>("castle_hip::linear_bwd");
    const auto s = ctx->get_saved_variables();
    const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
    auto [dx, dw] = op.call(g[0], s[0], s[1], need_x, need_w);
    return {need_x ? dx : Tensor(), need_w ? dw : Tensor()};
  }
};
std::tuple<Tensor, Tensor> linear_bwd_autograd(const Tensor& dy, const Tensor& x, const Tensor& weight, bool need_x, bool need_w) {
  static const auto op = op_handle<decltype(linear_bwd_op)>("castle_hip::linear_bwd");
  const bool graph = wants_graph({dy, x, weight});
  const at::AutoDispatchBelowADInplaceOrView below;
  const auto [dx, dw] = op.call(dy, x, weight, need_x, need_w);
  if (!graph) return {dx, dw};
  const auto r = no_second_derivatives({dx, dw});
  return {r[0], r[1]};
}
Tensor linear_autograd(const Tensor& x, const Tensor& weight) {
  if (!wants_graph({x, weight})) {
    static const auto op = op_handle<decltype(linear_op)>("castle_hip::linear");
    const at::AutoDispatchBelowADInplaceOrView below;
    return op.call(x, weight);
  }
  return LinearFn::apply(x, weight);
}

// ---- a whole layer over sequences ------------------------------------------------------------------------------
// [sum with the previous block's output] -> [RMS norm] -> fused projection -> attention core -> output projection, and
// its backward pass, as one autograd node: the modules one by one cost more host time than the kernels of a short
// sequence take.  With `delta` the layer works on x + delta and returns that sum too: a block of a residual stream.
struct LayerFn : torch::autograd::Function<LayerFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& delta, const std::optional<Tensor>& norm_w_,
                               const Tensor& w_qkv, const Tensor& w_out, std::optional<double> eps, int64_t heads, double scale, int64_t flags,
                               bool want_graph, bool keep_state, int64_t cache_rows, const std::vector<Tensor>& into = {}) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const Tensor norm_w = norm_w_.value_or(Tensor());
    const int64_t B = x.size(0), L = x.size(1), dim = x.size(2);
    const Tensor rows = x.reshape({B * L, dim});
    const Shape shape{(int)B, (int)heads, (int)L, (int)(w_qkv.size(0) / (6 * heads)), dtype_code(rows)};
    check_dims(shape.d, rows);
    Normed n;
    Tensor prepared, proj;
    if (!delta && norm_in_product(rows, norm_w, w_qkv)) {
      proj = project_packed_of_norm(rows, norm_w, eps, w_qkv, shape, want_graph, n, prepared);
    } else {
      n = norm_rows(rows, delta ? delta->reshape({B * L, dim}) : Tensor(), norm_w, eps, want_graph);
      proj = project_packed(n.h, w_qkv, shape, prepared);
    }
    proj = proj.view({B, L, w_qkv.size(0)});
    const bool want_U = cache_rows > 0;
    auto [merged, U, ws, state] = run_packed(proj, heads, scale, want_U, cache_rows, want_graph ? flags : flags | CASTLE_FLAG_FORWARD_ONLY, want_graph && keep_state, prepared, into.empty() ? Tensor() : into[0]);
    variable_list out{project(merged.view({B * L, merged.size(2)}), w_out).view({B, L, w_out.size(0)})};
    if (delta) out.push_back(n.sum.view({B, L, dim}));
    const size_t results = out.size();
    if (want_U) {   // the rows of the decode cache, behind U in the order of its fields: qu, kc, vc (rotated like the kernels use them)
      const Shape s = packed_shape(proj, heads);
      const int part[3] = {0, 4, 5};
      castle_view4 src[3], dst[3];
      out.push_back(U);
      for (int i = 0; i < 3; ++i) {
        out.push_back(into.empty() ? at::empty({B, heads, cache_rows, s.d}, proj.options()) : into[i + 1]);
        src[i] = packed_view(proj, s, 6, part[i]);
        dst[i] = view4(out.back());
      }
      check(castle_cache_rows(&src[0], &src[1], &src[2], &dst[0], &dst[1], &dst[2], s.B, s.H, s.L, s.d, s.dtype, (int)flags & CASTLE_FLAG_ROTARY,
                              stream_of(proj)), "castle_cache_rows");
    }
    if (want_graph) {
      // The layer's input itself is saved, not the rows that are a view of it: a view made below ADInplaceOrView has a
      // version of its own, so a change of the input in place would go unnoticed.  And only what the gradients asked for read:
      // anything else may be changed.
      const bool below = x.requires_grad() || (delta && delta->requires_grad()) || (norm_w.defined() && norm_w.requires_grad());
      const bool need_qkv = w_qkv.requires_grad();
      auto keep = [&](bool needed, const Tensor& t) { return !needed ? Tensor() : t.defined() && t.is_alias_of(x) ? x : t; };
      ctx->save_for_backward({keep(below && norm_w.defined(), n.sum), keep(below, norm_w), keep(below, w_qkv), keep(below || need_qkv, w_out),
                              keep(need_qkv, n.h), n.rstd, merged, ws, state});
      ctx->saved_data["heads"] = heads;
      ctx->saved_data["scale"] = scale;
      ctx->saved_data["flags"] = flags;
      ctx->mark_non_differentiable(variable_list(out.begin() + results, out.end()));
      ctx->set_materialize_grads(false);
    }
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (g[0].defined()) return once_differentiable([&] { return gradients(ctx, g); });
    variable_list grads(12);
    if (has_delta(g) && g[1].defined()) grads[0] = grads[1] = g[1];
    return grads;
  }
  // the results are y, the sum if there is a delta, and four cache tensors if they are asked for
  static bool has_delta(const variable_list& g) { return g.size() % 4 == 2; }
  static variable_list gradients(AutogradContext* ctx, const variable_list& g) {
    variable_list grads(12);
    const bool has_delta = LayerFn::has_delta(g);
    const Tensor dsum = has_delta ? g[1] : Tensor();
    const size_t nd = has_delta ? 1 : 0;   // needs_input_grad counts the tensors that were there
    const bool need_x = ctx->needs_input_grad(0) || (has_delta && ctx->needs_input_grad(1));
    const auto s = ctx->get_saved_variables();
    const Tensor &norm_w = s[1], &w_qkv = s[2], &w_out = s[3], &rstd = s[5], &merged = s[6], &ws = s[7], &state = s[8];
    const c10::DeviceGuard guard(merged.device());
    const int64_t B = merged.size(0), L = merged.size(1), heads = ctx->saved_data["heads"].toInt();
    const Tensor dy = g[0].reshape({B * L, g[0].size(2)});
    auto rows = [&](const Tensor& t) { return t.defined() && t.dim() == 3 ? t.reshape({B * L, t.size(2)}) : t; };
    const size_t nn = rstd.defined() ? 1 : 0;
    const bool need_norm = nn && ctx->needs_input_grad(1 + nd), need_qkv = ctx->needs_input_grad(1 + nd + nn);
    const bool need_core = need_x || need_norm || need_qkv, need_out = ctx->needs_input_grad(2 + nd + nn);
    const Tensor merged2 = merged.view({B * L, merged.size(2)});
    if (!need_core) {
      if (need_out) grads[4] = weight_grad(dy, merged2);
      return grads;
    }
    const Shape shape{(int)B, (int)heads, (int)L, (int)(merged.size(2) / heads), dtype_code(merged)};
    const int64_t flags = ctx->saved_data["flags"].toInt();
    Sums sums;
    Tensor dmerged, prepared;
    const bool both = need_out && own_projection_grads(dy, merged2, w_out, Tensor(), bwd_workspace_bytes(shape, flags, state), grads[4], dmerged, prepared, &sums);
    if (both) {
    } else if (own_product(dy, w_out, B * L, w_out.size(0), w_out.size(1), own_input_grad(w_out.size(0)))) {
      const Maxima m = maxima(dy, B * L, w_out.size(1), w_out.size(0), 0, w_out.size(1), bwd_workspace_bytes(shape, flags, state), false);
      prepared = m.prepared;
      dmerged = product(dy, false, w_out, true, CASTLE_GEMM_PLAIN, std::nullopt, m.get());
    } else {
      dmerged = at::mm(dy, w_out);
    }
    // (behind the product above, whose reads of dy it shares: before it, that one took 22 us instead of 16 for 16384 rows of 512)
    if (need_out && !both) grads[4] = weight_grad(dy, merged2, &sums);
    Tensor dproj = at::empty({B, L, 6 * merged.size(2)}, merged.options());
    castle_view4 d6[6];
    six_of_packed(dproj, shape, d6);
    // the backward kernels read the operand copies in the workspace: the projection itself is not kept
    run_bwd(d6, packed_view(merged, shape, 1, 0), packed_view(dmerged, shape, 1, 0), shape, ctx->saved_data["scale"].toDouble(), flags, d6, ws,
            state, prepared);
    const Tensor dp2 = dproj.view({B * L, dproj.size(2)});
    Tensor dh, none;
    const bool both_in = need_qkv && (need_x || need_norm) && own_projection_grads(dp2, rows(s[4]), w_qkv, Tensor(), -1, grads[3], dh, none, &sums);
    if (need_qkv && !both_in) grads[3] = weight_grad(dp2, rows(s[4]), &sums);
    if (need_x || need_norm) {
      auto [dx, dn] = norm_rows_bwd(both_in ? dh : input_grad(dp2, w_qkv), rows(s[0]), rstd, norm_w, rows(dsum), need_x, need_norm, &sums);
      if (need_norm) grads[2] = dn;
      if (need_x) grads[0] = dx.view({B, L, dx.size(1)});
      if (has_delta) grads[1] = grads[0];
    }
    sums.flush();
    return grads;
  }
};

// x (B, L, dim) -> [y, x + delta if there is a delta, then U, qu, kc, vc with buffers of `cache_rows` rows when cache_rows > 0]
variable_list layer_parallel(const Tensor& x, const std::optional<Tensor>& delta, const std::optional<Tensor>& norm_w, std::optional<double> eps,
                             const Tensor& w_qkv, const Tensor& w_out, int64_t heads, double scale, int64_t flags, bool keep_state, int64_t cache_rows) {
  const c10::DeviceGuard guard(x.device());
  if (!wants_graph({x, delta.value_or(Tensor()), norm_w.value_or(Tensor()), w_qkv, w_out}))
    return LayerFn::forward(nullptr, x, delta, norm_w, w_qkv, w_out, eps, heads, scale, flags, false, false, cache_rows);
  return LayerFn::apply(x, delta, norm_w, w_qkv, w_out, eps, heads, scale, flags, true, keep_state, cache_rows);
}

// The same into the four buffers of a decode cache that is there already, without a graph -> [y, x + delta if there is a delta]
variable_list layer_prefill(const Tensor& x, const std::optional<Tensor>& delta, const std::optional<Tensor>& norm_w, std::optional<double> eps,
                            const Tensor& w_qkv, const Tensor& w_out, int64_t heads, double scale, int64_t flags, const std::vector<Tensor>& buffers) {
  const c10::DeviceGuard guard(x.device());
  TORCH_CHECK_VALUE(buffers.size() == 4 && x.dim() == 3 && !wants_graph({x, delta.value_or(Tensor()), norm_w.value_or(Tensor()), w_qkv, w_out}),
                    "layer_prefill: four buffers, and no gradients");
  const int64_t d = w_qkv.size(0) / (6 * heads), rows = buffers[0].dim() == 4 ? buffers[0].size(2) : 0;
  for (const Tensor& t : buffers)
    TORCH_CHECK_VALUE(t.is_contiguous() && t.sizes() == at::IntArrayRef({x.size(0), heads, rows, d}) && rows >= x.size(1) && t.scalar_type() == x.scalar_type() &&
                      t.device() == x.device(), "layer_prefill: unexpected buffers");
  auto out = LayerFn::forward(nullptr, x, delta, norm_w, w_qkv, w_out, eps, heads, scale, flags, false, false, rows, buffers);
  out.resize(delta ? 2 : 1);
  return out;
}

// ---- the other blocks of a language model over sequences ---------------------------------------------------------
// Feed-forward block of a residual stream: s = x + delta, y = gelu(norm(s) w_up^T) w_down^T -> [y, s]
struct FeedForwardFn : torch::autograd::Function<FeedForwardFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& delta, const Tensor& norm_w, const Tensor& w_up,
                               const Tensor& w_down, std::optional<double> eps, bool want_graph) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const int64_t R = x.numel() / x.size(-1);
    const Normed n = norm_rows(x.reshape({R, x.size(-1)}), delta.reshape({R, x.size(-1)}), norm_w, eps, want_graph);
    Tensor up, act;
    if (own_product(n.h, w_up, R, w_up.size(0), w_up.size(1), own_forward(w_up.size(1)))) {   // GELU on the way out
      act = at::empty({R, w_up.size(0)}, n.h.options());
      up = product(n.h, false, w_up, false, CASTLE_GEMM_GELU, act);
    } else {
      up = at::mm(n.h, w_up.t());
      act = at::gelu(up);
    }
    Tensor y = project(act, w_down).view(x.sizes());
    if (want_graph) {
      ctx->save_for_backward({n.sum, norm_w, w_up, w_down, n.h, n.rstd, up, act});
      ctx->set_materialize_grads(false);
    }
    return {y, n.sum.view(x.sizes())};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (g[0].defined()) return once_differentiable([&] { return gradients(ctx, g); });
    variable_list grads(7);
    if (g[1].defined()) grads[0] = grads[1] = g[1];
    return grads;
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& g) {
    variable_list grads(7);
    const Tensor dsum = g[1];
    const bool need_x = ctx->needs_input_grad(0) || ctx->needs_input_grad(1), need_norm = ctx->needs_input_grad(2), need_up = ctx->needs_input_grad(3);
    const auto s = ctx->get_saved_variables();
    const Tensor &sum = s[0], &norm_w = s[1], &w_up = s[2], &w_down = s[3], &h = s[4], &rstd = s[5], &up = s[6], &act = s[7];
    const c10::DeviceGuard guard(h.device());
    const int64_t R = sum.size(0), dim = sum.size(1);
    const Tensor dy = g[0].reshape({R, dim});
    const bool below = need_x || need_norm || need_up, need_down = ctx->needs_input_grad(4);
    Sums sums;
    Tensor dup, dh, none;
    const bool both = below && need_down && own_projection_grads(dy, act, w_down, up, -1, grads[4], dup, none, &sums);
    if (need_down && !both) grads[4] = weight_grad(dy, act, below ? &sums : nullptr);
    if (!below) return grads;
    if (!both)
      dup = own_product(dy, w_down, R, dim, w_down.size(1), kOwnGeluSlope) ? product(dy, false, w_down, true, CASTLE_GEMM_GELU_SLOPE, up)
                                                                           : at::gelu_backward(at::mm(dy, w_down), up);
    const bool both_up = need_up && (need_x || need_norm) && own_projection_grads(dup, h, w_up, Tensor(), -1, grads[3], dh, none, &sums);
    if (need_up && !both_up) grads[3] = weight_grad(dup, h, &sums);
    if (need_x || need_norm) {
      auto [dx, dn] = norm_rows_bwd(both_up ? dh : input_grad(dup, w_up), sum, rstd, norm_w, dsum.defined() ? dsum.reshape({R, dim}) : Tensor(), need_x, need_norm, &sums);
      if (need_norm) grads[2] = dn;
      if (need_x) grads[0] = grads[1] = dx.view(g[0].sizes());
    }
    sums.flush();
    return grads;
  }
};

variable_list feed_forward(const Tensor& x, const Tensor& delta, const Tensor& norm_w, std::optional<double> eps, const Tensor& w_up, const Tensor& w_down) {
  const c10::DeviceGuard guard(x.device());
  if (!wants_graph({x, delta, norm_w, w_up, w_down})) return FeedForwardFn::forward(nullptr, x, delta, norm_w, w_up, w_down, eps, false);
  return FeedForwardFn::apply(x, delta, norm_w, w_up, w_down, eps, true);
}

// norm(x + delta) w^T: the end of a residual stream
struct HeadFn : torch::autograd::Function<HeadFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& delta, const Tensor& norm_w, const Tensor& w, std::optional<double> eps,
                        bool want_graph) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const int64_t B = x.size(0), L = x.size(1), dim = x.size(2);
    const Normed n = norm_rows(x.reshape({B * L, dim}), delta.reshape({B * L, dim}), norm_w, eps, want_graph);
    if (want_graph) ctx->save_for_backward({n.sum, norm_w, w, n.h, n.rstd});
    return project(n.h, w).view({B, L, w.size(0)});
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return once_differentiable([&] { return gradients(ctx, g); });
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& g) {
    variable_list grads(6);
    const auto s = ctx->get_saved_variables();
    const Tensor &sum = s[0], &norm_w = s[1], &w = s[2], &h = s[3], &rstd = s[4];
    const c10::DeviceGuard guard(h.device());
    const Tensor dy = g[0].reshape({sum.size(0), w.size(0)});
    const bool need_x = ctx->needs_input_grad(0) || ctx->needs_input_grad(1), need_norm = ctx->needs_input_grad(2);
    const bool need_w = ctx->needs_input_grad(3);
    Sums sums;
    Tensor dh, none;
    const bool both = need_w && (need_x || need_norm) && own_projection_grads(dy, h, w, Tensor(), -1, grads[3], dh, none, &sums);
    if (need_w && !both) grads[3] = weight_grad(dy, h, &sums);
    if (need_x || need_norm) {
      auto [dx, dn] = norm_rows_bwd(both ? dh : input_grad(dy, w), sum, rstd, norm_w, Tensor(), need_x, need_norm, &sums);
      if (need_norm) grads[2] = dn;
      if (need_x) grads[0] = grads[1] = dx.view({g[0].size(0), g[0].size(1), sum.size(1)});
    }
    sums.flush();
    return grads;
  }
};

Tensor head(const Tensor& x, const Tensor& delta, const Tensor& norm_w, std::optional<double> eps, const Tensor& w) {
  const c10::DeviceGuard guard(x.device());
  if (!wants_graph({x, delta, norm_w, w})) return HeadFn::forward(nullptr, x, delta, norm_w, w, eps, false);
  return HeadFn::apply(x, delta, norm_w, w, eps, true);
}

// a (B, n) tensor of token numbers as the kernels address it
Tensor token_rows(const Tensor& t) { return t.stride(1) == 1 || t.size(1) == 1 ? t : t.contiguous(); }

// mean cross entropy of (B, n, V) logits against (B, n) classes; one launch pair where the library's operator on the
// transposed logits takes 190 us forward and 180 back at 16384 x 256
struct CrossEntropyFn : torch::autograd::Function<CrossEntropyFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits_, const Tensor& target_, bool want_graph) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const Tensor logits = row_major(logits_), target = token_rows(target_);
    const int64_t V = logits.size(2), R = logits.numel() / V;
    const auto f = logits.options().dtype(at::kFloat);
    Tensor loss = at::empty({}, logits.options()), lse = at::empty({R}, f), inv = at::empty({}, f), ws = bytes(CASTLE_CROSS_ENTROPY_WORKSPACE, logits);
    check(castle_cross_entropy(logits.data_ptr(), static_cast<const int64_t*>(target.data_ptr()), target.size(1), target.stride(0), R, (int)V, loss.data_ptr(),
                               static_cast<float*>(lse.data_ptr()), static_cast<float*>(inv.data_ptr()), dtype_code(logits), ws.data_ptr(), ws.numel(),
                               stream_of(logits)),
          "castle_cross_entropy");
    if (want_graph) ctx->save_for_backward({logits, target, lse, inv});
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return once_differentiable([&] { return gradients(ctx, g); });
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &logits = s[0], &target = s[1], &lse = s[2], &inv = s[3];
    const c10::DeviceGuard guard(logits.device());
    Tensor d = at::empty_like(logits);
    const int64_t V = logits.size(2);
    check(castle_cross_entropy_bwd(logits.data_ptr(), static_cast<const int64_t*>(target.data_ptr()), target.size(1), target.stride(0), logits.numel() / V,
                                   (int)V, static_cast<const float*>(lse.data_ptr()), static_cast<const float*>(inv.data_ptr()), g[0].data_ptr(), d.data_ptr(),
                                   dtype_code(logits), stream_of(logits)),
          "castle_cross_entropy_bwd");
    return {d, Tensor(), Tensor()};
  }
};

Tensor cross_entropy(const Tensor& logits, const Tensor& target) {
  const c10::DeviceGuard guard(logits.device());
  TORCH_CHECK_VALUE(target.dim() == 2 && target.scalar_type() == at::kLong && target.device() == logits.device() && logits.dim() == 3 &&
                        target.size(0) == logits.size(0) && target.size(1) == logits.size(1), "cross_entropy: unexpected target");
  if (logits.size(2) * logits.element_size() % 16 != 0 || logits.numel() == 0) return at::cross_entropy_loss(logits.transpose(1, 2), target);
  if (!wants_graph({logits})) return CrossEntropyFn::forward(nullptr, logits, target, false);
  return CrossEntropyFn::apply(logits, target, true);
}

// the token embedding, with a gradient that needs neither a sort nor the host where the vocabulary is small
struct EmbeddingFn : torch::autograd::Function<EmbeddingFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& weight, const Tensor& index) {
    const at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({index});
    ctx->saved_data["vocabulary"] = weight.size(0);
    return at::embedding(weight, index);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return once_differentiable([&] { return gradients(ctx, g); });
  }
  static variable_list gradients(AutogradContext* ctx, const variable_list& g) {
    const Tensor index = token_rows(ctx->get_saved_variables()[0]);
    const c10::DeviceGuard guard(index.device());
    const int64_t V = ctx->saved_data["vocabulary"].toInt(), D = g[0].size(-1), R = index.numel();
    const int64_t nbytes = castle_embedding_grad_workspace_bytes(R, (int)V, (int)D, dtype_code(g[0]));
    if (nbytes < 0 || V * D % 8 != 0) return {at::embedding_dense_backward(g[0], index, V, -1, false), Tensor()};
    const Tensor dy = row_major(g[0]);
    Tensor dw = at::empty({V, D}, dy.options()), ws = bytes(nbytes, dy);
    check(castle_embedding_grad(dy.data_ptr(), static_cast<const int64_t*>(index.data_ptr()), index.size(1), index.stride(0), R, (int)V, (int)D, dw.data_ptr(),
                                dtype_code(dy), ws.data_ptr(), nbytes, stream_of(dy)),
          "castle_embedding_grad");
    return {dw, Tensor()};
  }
};

Tensor embedding(const Tensor& weight, const Tensor& index) {
  const c10::DeviceGuard guard(weight.device());
  if (!wants_graph({weight}) || index.numel() == 0) return at::embedding(weight, index);
  return EmbeddingFn::apply(weight, index);
}

// ---- the cached single-token step ------------------------------------------------------------------------------
// rows of a matrix that the kernels can read 16 bytes at a time
bool rows_readable(const Tensor& t) {
  return t.dim() == 2 && t.stride(1) == 1 && t.stride(0) % (16 / t.element_size()) == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// (B, 1, K) x (N, K) through the small-M kernel: see castle_small_linear_fused
Tensor small_linear(const Tensor& x, const Tensor& w, const std::optional<Tensor>& norm_w, double eps, int64_t act,
                    const std::optional<Tensor>& residual) {
  const c10::DeviceGuard guard(x.device());
  no_tangent(x);
  const int64_t B = x.size(0), N = w.size(0);
  Tensor y = at::empty({B, 1, N}, x.options());
  check(castle_small_linear_fused(x.data_ptr(), w.data_ptr(), y.data_ptr(), (int)B, (int)N, (int)x.size(2), x.stride(0), w.stride(0), N,
                                  dtype_code(x), norm_w ? norm_w->data_ptr() : nullptr, (float)eps, (int)act,
                                  residual ? residual->data_ptr() : nullptr, residual ? residual->stride(0) : 0, stream_of(x)),
        "castle_small_linear_fused");
  return y;
}

// logits (B, V) -> one token per row into `token` (B,) (any stride) and, if given, `copy` (B,) contiguous
void sample_tokens(const Tensor& logits, const std::optional<Tensor>& uniform, int64_t k, double temperature, const Tensor& token,
                   const std::optional<Tensor>& copy) {
  const c10::DeviceGuard guard(logits.device());
  TORCH_CHECK_VALUE(logits.is_cuda() && logits.dim() == 2 && logits.stride(1) == 1 && token.scalar_type() == at::kLong && token.dim() == 1 &&
                        token.size(0) == logits.size(0) && token.device() == logits.device(), "sample_tokens: unexpected logits or token tensor");
  TORCH_CHECK_VALUE(!uniform || (uniform->is_contiguous() && uniform->scalar_type() == at::kFloat && uniform->sizes() == logits.sizes()),
                    "sample_tokens: unexpected uniform numbers");
  TORCH_CHECK_VALUE(!copy || (copy->is_contiguous() && copy->scalar_type() == at::kLong && copy->numel() == logits.size(0)),
                    "sample_tokens: unexpected copy");
  check(castle_sample(logits.data_ptr(), logits.stride(0), uniform ? static_cast<const float*>(uniform->data_ptr()) : nullptr,
                      (int)logits.size(0), (int)logits.size(1), (int)k, 1.f / (float)temperature, static_cast<int64_t*>(token.data_ptr()),
                      token.stride(0), copy ? static_cast<int64_t*>(copy->data_ptr()) : nullptr, dtype_code(logits), stream_of(logits)),
        "castle_sample");
}

// embedding of one token per row: (V, K) table, (B, 1) tokens -> (B, 1, K)
Tensor gather_rows(const Tensor& table, const Tensor& index) {
  const c10::DeviceGuard guard(table.device());
  if (!rows_readable(table) || table.size(1) % (16 / table.element_size()) != 0 || !index.is_contiguous()) return at::embedding(table, index);
  Tensor y = at::empty({index.size(0), 1, table.size(1)}, table.options());
  check(castle_gather_rows(table.data_ptr(), table.size(0), table.stride(0), (int)table.size(1), static_cast<const int64_t*>(index.data_ptr()),
                           (int)index.numel(), y.data_ptr(), dtype_code(table), stream_of(table)),
        "castle_gather_rows");
  return y;
}

// The capacity buffers of one decode cache with everything a step needs to know about them
class StepPlan {
 public:
  StepPlan(std::vector<Tensor> buffers, Tensor ring, Tensor gates, Tensor workspace, bool u_half)
      : buffers_(std::move(buffers)), ring_(std::move(ring)), gates_(std::move(gates)), workspace_(std::move(workspace)) {
    TORCH_CHECK(buffers_.size() == 4 && gates_.scalar_type() == at::kFloat && gates_.is_contiguous(), "StepPlan: unexpected buffers");
    for (int i = 0; i < 4; ++i) views_[i] = view4(buffers_[i]);
    s_ = shape_of(buffers_[0]);   // L = capacity
    flags_ = u_half ? CASTLE_FLAG_U_HALF : 0;
    deferred_ = {view4(ring_), view4(gates_), 0, nullptr};
  }

  // proj (B, 1, 6 H d) -> (B, 1, H d) at row count t.  base >= 0: deferred write-back of the lookahead keys from
  // that row count on (see castle_deferred); base < 0: every step writes them.  With t_device (and base_device) the
  // row counts are read by the kernels, as a captured graph of the step needs it.
  Tensor attend(const Tensor& proj_, int64_t t, int64_t base, double scale, bool rotary, const std::optional<Tensor>& t_device,
                const std::optional<Tensor>& base_device) {
    check_count(t, t_device);
    no_tangent(proj_);
    const Tensor proj = packed_readable(proj_);
    TORCH_CHECK_VALUE(proj.dim() == 3 && proj.size(0) == s_.B && proj.size(1) == 1 && proj.size(2) == 6LL * s_.H * s_.d &&
                          proj.scalar_type() == buffers_[0].scalar_type() && proj.device() == buffers_[0].device(),
                      "the projection does not belong to this cache");
    const c10::DeviceGuard guard(proj.device());
    Tensor out = at::empty({s_.B, 1, (int64_t)s_.H * s_.d}, proj.options());
    Shape one = s_;
    one.L = 1;
    castle_view4 v[6];
    six_of_packed(proj, one, v);
    const castle_view4 vo = packed_view(out, one, 1, 0), *c = views_;
    castle_deferred def = deferred(base, base_device);
    const castle_deferred* pd = base >= 0 || base_device ? &def : nullptr;
    const int flags = flags_ | (rotary ? CASTLE_FLAG_ROTARY : 0);
    used_on_current_stream();
    void* ws = workspace_.data_ptr();
    const int64_t wb = workspace_.numel();
    check(t_device ? castle_decode_step_device_count(c, c + 1, c + 2, c + 3, count_ptr(t_device), s_.L, &v[0], &v[1], &v[2], &v[3], &v[4], &v[5],
                                                     s_.B, s_.H, s_.d, s_.dtype, (float)scale, flags, &vo, pd, ws, wb, stream_of(proj))
                   : castle_decode_step(c, c + 1, c + 2, c + 3, (int)t, s_.L, &v[0], &v[1], &v[2], &v[3], &v[4], &v[5], s_.B, s_.H, s_.d,
                                        s_.dtype, (float)scale, flags, &vo, pd, ws, wb, stream_of(proj)),
          "castle_decode_step");
    return out;
  }

  // the steps of this cache are part of a loop over more cached rows than the last-level cache holds
  void read_once(bool on) { flags_ = on ? flags_ | CASTLE_FLAG_READ_ONCE : flags_ & ~CASTLE_FLAG_READ_ONCE; }

  // the whole layer for one token: x (B, 1, dim) -> (B, 1, dim), plus `residual` if there is one
  Tensor layer(const Tensor& x, const std::optional<Tensor>& norm_w, std::optional<double> eps, const Tensor& w_qkv, const Tensor& w_out,
               int64_t max_rows, int64_t t, int64_t base, double scale, bool rotary, const std::optional<Tensor>& residual,
               const std::optional<Tensor>& t_device, const std::optional<Tensor>& base_device) {
    const int64_t B = s_.B, dim = x.size(-1), inner = (int64_t)s_.H * s_.d;
    const c10::DeviceGuard guard(x.device());
    check_count(t, t_device);
    no_tangent(x);
    TORCH_CHECK_VALUE(x.dim() == 3 && x.size(0) == B && x.size(1) == 1 && w_qkv.dim() == 2 && w_qkv.size(0) == 6 * inner && w_qkv.size(1) == dim &&
                          w_out.dim() == 2 && w_out.size(1) == inner && x.scalar_type() == buffers_[0].scalar_type() && x.device() == buffers_[0].device(),
                      "the token or the weights do not belong to this cache");
    if (B > max_rows || w_out.size(0) != dim || !rows_readable(w_qkv) || !rows_readable(w_out)) {
      const Tensor proj = at::linear(norm_w ? at::rms_norm(x, {dim}, norm_w, eps) : x, w_qkv);
      const Tensor y = at::linear(attend(proj, t, base, scale, rotary, t_device, base_device), w_out);
      return residual ? *residual + y : y;
    }
    const Tensor xr = rows_readable(x.select(1, 0)) ? x : x.contiguous();
    const Tensor nw = norm_w ? norm_w->contiguous() : Tensor();
    const Tensor res = residual ? (residual->stride(2) == 1 ? *residual : residual->contiguous()) : Tensor();
    const double e = norm_eps(eps);
    // the projection is scratch of the step like the workspace: kept with it, an allocation costs more than a microsecond
    if (!proj_.defined()) proj_ = at::empty({B, 6 * inner}, x.options().requires_grad(false));
    // For the step as one launch, where it is one.  Not while a graph is recorded: the zeros would be there only once it is replayed, and
    // steps outside of it use the words too.
    const bool once = !t_device && castle_decode_layer_once_ok(s_.B, s_.H, s_.d, s_.dtype, (int)t, (int)dim);
    if (once && !control_.defined() && c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None) {
      const int64_t n = check(castle_decode_layer_control_bytes(s_.B, s_.H, s_.d, s_.dtype), "castle_decode_layer_control_bytes");
      control_ = at::zeros({n}, x.options().dtype(at::kByte).requires_grad(false));
    }
    const bool words = once && control_.defined();
    used_on_current_stream();
    Tensor y = at::empty({B, 1, dim}, x.options());
    const castle_view4* c = views_;
    castle_deferred def = deferred(base, base_device);
    check(castle_decode_layer_once(c, c + 1, c + 2, c + 3, (int)t, t_device ? count_ptr(t_device) : nullptr, s_.L, xr.data_ptr(), xr.stride(0), (int)dim,
                              nw.defined() ? nw.data_ptr() : nullptr, (float)e, w_qkv.data_ptr(), w_qkv.stride(0), w_out.data_ptr(),
                              w_out.stride(0), res.defined() ? res.data_ptr() : nullptr, res.defined() ? res.stride(0) : 0, y.data_ptr(), dim,
                              proj_.data_ptr(), s_.B, s_.H, s_.d, s_.dtype, (float)scale, flags_ | (rotary ? CASTLE_FLAG_ROTARY : 0),
                              base >= 0 || base_device ? &def : nullptr, workspace_.data_ptr(), workspace_.numel(), words ? control_.data_ptr() : nullptr,
                              words ? control_.numel() : 0, stream_of(x)),
          "castle_decode_layer_once");
    return y;
  }

 private:
  // What the steps work on was allocated on the stream of the prompt or of the first step; the allocator has to know of every other
  // stream that uses it, or it hands the memory of a dropped cache out again before a step on that stream is through.
  void used_on_current_stream() {
    const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(buffers_[0].get_device());
    if (stream_ && *stream_ == stream && recorded_proj_ == proj_.defined() && recorded_control_ == control_.defined()) return;
    // (straight to the allocator: record_stream costs a microsecond a tensor)
    auto record = [&](const Tensor& t) {
      if (t.defined()) c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::recordStreamMasqueradingAsCUDA(t.storage().data_ptr(), stream);
    };
    for (const Tensor& t : buffers_) record(t);
    for (const Tensor* t : {&ring_, &gates_, &workspace_, &proj_, &control_}) record(*t);
    stream_ = stream;
    recorded_proj_ = proj_.defined();
    recorded_control_ = control_.defined();
  }
  static const int32_t* count_ptr(const std::optional<Tensor>& t) { return static_cast<const int32_t*>(t->data_ptr()); }
  void check_count(int64_t t, const std::optional<Tensor>& t_device) const {
    if (t_device) {
      TORCH_CHECK_VALUE(t_device->scalar_type() == at::kInt && t_device->numel() == 1 && t_device->device() == buffers_[0].device(),
                        "t_device must be a one-element int32 tensor on the GPU of the step");
      return;
    }
    TORCH_CHECK_VALUE(t >= 0 && t < s_.L, "cache capacity ", s_.L, " cannot take row ", t);
  }
  castle_deferred deferred(int64_t base, const std::optional<Tensor>& base_device) const {
    castle_deferred r = deferred_;
    r.base = (int)std::max<int64_t>(base, 0);
    r.base_device = base_device ? count_ptr(base_device) : nullptr;
    return r;
  }

  std::vector<Tensor> buffers_;
  Tensor ring_, gates_, workspace_, proj_, control_;
  std::optional<c10::hip::HIPStreamMasqueradingAsCUDA> stream_;   // of the last step
  bool recorded_proj_ = false, recorded_control_ = false;
  castle_view4 views_[4];
  castle_deferred deferred_;
  Shape s_;
  int flags_;
};

}  // namespace

TORCH_LIBRARY(castle_hip, m) {
  m.set_python_module("lookahead_keys_attention_amd.ops");   // the fake (meta) implementations live there
  const std::vector<at::Tag> tags = {at::Tag::pt2_compliant_tag};
  m.def("attention(Tensor q, Tensor k, Tensor v, Tensor qu, Tensor ku, Tensor vu, float scale, bool want_U, int flags, bool keep_state) "
        "-> (Tensor, Tensor, Tensor, Tensor)", tags);
  m.def("attention_bwd(Tensor q, Tensor k, Tensor v, Tensor qu, Tensor ku, Tensor vu, Tensor out, Tensor dout, Tensor ws, Tensor state, "
        "float scale, int flags) -> Tensor", tags);
  m.def("attention_packed(Tensor proj, int heads, float scale, bool want_U, int row_capacity, int flags, bool keep_state) "
        "-> (Tensor, Tensor, Tensor, Tensor)", tags);
  m.def("attention_packed_bwd(Tensor proj, Tensor merged, Tensor dmerged, Tensor ws, Tensor state, int heads, float scale, int flags) "
        "-> Tensor", tags);
  m.def("rms_norm(Tensor x, Tensor weight, float? eps) -> (Tensor, Tensor)", tags);
  m.def("rms_norm_bwd(Tensor dh, Tensor x, Tensor rstd, Tensor weight, bool need_x=True, bool need_w=True) -> (Tensor, Tensor)", tags);
  m.def("linear(Tensor x, Tensor weight) -> Tensor", tags);
  m.def("linear_bwd(Tensor dy, Tensor x, Tensor weight, bool need_x=True, bool need_w=True) -> (Tensor, Tensor)", tags);
}
TORCH_LIBRARY_IMPL(castle_hip, CUDA, m) {
  m.impl("attention", &attention);
  m.impl("attention_bwd", &attention_bwd);
  m.impl("attention_packed", &attention_packed);
  m.impl("attention_packed_bwd", &attention_packed_bwd);
  m.impl("rms_norm", &rms_norm_op);
  m.impl("rms_norm_bwd", &rms_norm_bwd_op);
  m.impl("linear", &linear_op);
  m.impl("linear_bwd", &linear_bwd_op);
}
// CPU tensors: an error that says what is wrong
TORCH_LIBRARY_IMPL(castle_hip, CPU, m) {
  m.impl("attention", &attention);
  m.impl("attention_packed", &attention_packed);
}
TORCH_LIBRARY_IMPL(castle_hip, Autograd, m) {
  m.impl("attention", &attention_autograd);
  m.impl("attention_packed", &attention_packed_autograd);
  m.impl("attention_bwd", &attention_bwd_autograd);
  m.impl("attention_packed_bwd", &attention_packed_bwd_autograd);
  m.impl("rms_norm", &rms_norm_autograd);
  m.impl("rms_norm_bwd", &rms_norm_bwd_autograd);
  m.impl("linear", &linear_autograd);
  m.impl("linear_bwd", &linear_bwd_autograd);
}

PYBIND11_MODULE(_castle_host, m) {
  namespace py = pybind11;
  m.attr("ABI_VERSION") = castle_abi_version();
  using unlocked = py::call_guard<py::gil_scoped_release>;
  m.def("layer_parallel", &layer_parallel, unlocked());
  m.def("layer_prefill", &layer_prefill, unlocked());
  m.def("product", [](const Tensor& a, bool a_t, const Tensor& b, bool b_t, int64_t epilogue, const std::optional<Tensor>& aux) {
    return product(a, a_t, b, b_t, epilogue, aux);
  }, unlocked());
  m.def("feed_forward", &feed_forward, unlocked());
  m.def("head", &head, unlocked());
  m.def("cross_entropy", &cross_entropy, unlocked());
  m.def("embedding", &embedding, unlocked());
  m.def("small_linear", &small_linear, unlocked());
  m.def("sample_tokens", &sample_tokens, unlocked());
  m.def("gather_rows", &gather_rows, unlocked());
  py::class_<StepPlan>(m, "StepPlan")
      .def(py::init<std::vector<Tensor>, Tensor, Tensor, Tensor, bool>())
      .def("attend", &StepPlan::attend, unlocked())
      .def("read_once", &StepPlan::read_once)
      .def("layer", &StepPlan::layer, unlocked());
}
