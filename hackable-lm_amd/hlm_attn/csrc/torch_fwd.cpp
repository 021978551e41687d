// Host work of plain eager calls in C++: check, allocate through torch's
// caching allocator, launch through the C ABI (include/hlm_attn.h).  Host code
// only, linked against libhlm_attn.so in the same directory.
//
// * fwd: the no-grad attention forward of the evaluation harness's calls
//   (lm_eval_hackable_lm.py:134-160,185-207: batch 1, ragged T, one full
//   forward per token).  At batch 1 and short T the kernel takes a few
//   microseconds, so the host work around the launch decides the call rate;
//   done in Python it costs about twice the launch.
// * attn_train, qk_norm_rope_train, residual_rms_norm_train: the
//   differentiable calls of a training step as C++ autograd functions.  The
//   Python custom ops that they stand for cost 70-170 us of host time per
//   forward and backward, as much as or more than the kernels of a layer.  The
//   caller (ops.eager_ext) uses them only where no tracing, dispatch or function
//   mode, function transform or forward-mode AD is active; a backward that runs
//   under one of these, or with create_graph, calls the custom op itself.
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <strings.h>

#include <cstdint>
#include <cstdlib>
#include <optional>
#include <tuple>
#include <vector>

#include "../../../include/hlm_attn.h"

namespace {

// The kernels' layout: (B, T, H, D) with unit D stride, (batch, time, head)
// strides multiples of 8 elements, rows that do not overlap, 16-byte aligned.
bool kernel_ready(const at::Tensor& t) {
  const auto s = t.strides();
  return s[3] == 1 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 && s[0] >= 0 && s[1] >= 0 && s[2] >= 0 &&
         s[1] >= t.size(3) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// q, k, v are bf16 (B, T, H, D) tensors on one device with the kernels' layout.
bool takes(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t window) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
  if (q.scalar_type() != at::kBFloat16 || k.scalar_type() != at::kBFloat16 || v.scalar_type() != at::kBFloat16)
    return false;
  if (!q.is_cuda() || k.device() != q.device() || v.device() != q.device()) return false;
  if (k.sizes() != v.sizes() || q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3) ||
      k.size(2) == 0 || q.size(2) % k.size(2) != 0)
    return false;
  if (!kernel_ready(q) || !kernel_ready(k) || !kernel_ready(v)) return false;
  return q.size(0) <= INT32_MAX && q.size(1) <= INT32_MAX && q.size(2) <= INT32_MAX && q.size(3) <= INT32_MAX &&
         window >= 0 && window <= INT32_MAX;
}

// Returns {o, lse}, or an empty list when the inputs are not such tensors (the
// caller then takes its general path, which converts or raises).  A launch
// error raises with the C ABI's message.
std::vector<at::Tensor> fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t window,
                            double scale, int64_t stream) {
  if (!takes(q, k, v, window)) return {};
  const int64_t B = q.size(0), T = q.size(1), H = q.size(2), Hkv = k.size(2), D = q.size(3);
  const c10::DeviceGuard guard(q.device());
  at::Tensor o = at::empty({B, T, H, D}, q.options());
  at::Tensor lse = at::empty({B, H, T}, q.options().dtype(at::kFloat));
  const int nsplit = hlm_attn_fwd_split_count((int)B, (int)T, (int)H, (int)D, (int)window);
  const int64_t so[3] = {T * H * D, H * D, D};
  const auto sq = q.strides(), sk = k.strides(), sv = v.strides();
  const int64_t sq3[3] = {sq[0], sq[1], sq[2]}, sk3[3] = {sk[0], sk[1], sk[2]}, sv3[3] = {sv[0], sv[1], sv[2]};
  void* st = reinterpret_cast<void*>(static_cast<uintptr_t>(stream));
  int rc;
  if (nsplit > 1) {
    at::Tensor ws = at::empty({nsplit * B * H * T * (D + 2)}, q.options().dtype(at::kFloat));
    rc = hlm_attn_fwd_split(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                            ws.data_ptr<float>(), nsplit, (int)B, (int)T, (int)H, (int)Hkv, (int)D, sq3, sk3, sv3, so,
                            (int)window, (float)scale, st);
  } else {
    rc = hlm_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), (int)B, (int)T,
                      (int)H, (int)Hkv, (int)D, sq3, sk3, sv3, so, (int)window, (float)scale, st);
  }
  TORCH_CHECK(rc == 0, "hip attention failed (code ", rc, "): ", hlm_attn_last_error());
  return {o, lse};
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The current stream of the tensor's device, as the backward finds it: the
// autograd engine runs a node on the stream of its forward.
void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// A tensor whose memory may be handed to a kernel as it is: strided, on a ROCm
// device, no wrapper of a transform or mode around it.
bool plain(const at::Tensor& t) {
  static constexpr c10::DispatchKeySet kWrapped(
      {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched, c10::DispatchKey::Functionalize,
       c10::DispatchKey::ZeroTensor, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kWrapped);
}

// Whether a backward must go through its custom op: create_graph (the op then
// refuses a second derivative), a dispatch or function mode, or a wrapped
// gradient.
bool needs_op(const variable_list& ts) {
  if (at::GradMode::is_enabled() || c10::impl::TorchDispatchModeTLS::stack_len() > 0 ||
      at::impl::PythonTorchFunctionTLS::stack_len() > 0)
    return true;
  for (const auto& t : ts)
    if (!plain(t)) return true;
  return false;
}

// Calls torch.ops.hackable_lm.<name>, through Python: function modes see only
// calls that are made there.
template <class... Args>
variable_list call_op(const char* name, Args&&... args) {
  const py::gil_scoped_acquire gil;
  const py::object op = py::module_::import("torch").attr("ops").attr("hackable_lm").attr(name).attr("default");
  const py::object out = op(std::forward<Args>(args)...);
  if (py::isinstance<py::tuple>(out)) return out.cast<variable_list>();
  return {out.cast<at::Tensor>()};
}

void check(int rc) { TORCH_CHECK(rc == 0, "hip attention failed (code ", rc, "): ", hlm_attn_last_error()); }

struct Strides {
  int64_t s[3];
  explicit Strides(const at::Tensor& t) : s{t.stride(0), t.stride(1), t.stride(2)} {}
};

// A (B, T, heads, D) tensor of the backward in the kernels' layout.
at::Tensor rows4(at::Tensor t, at::IntArrayRef sizes, c10::Device device) {
  TORCH_CHECK(t.device() == device && t.sizes() == sizes, "a tensor of the backward does not match the forward's");
  if (t.scalar_type() != at::kBFloat16) t = t.to(at::kBFloat16);
  return kernel_ready(t) ? t : t.contiguous();
}

bool fused_backward_selected() {
  const char* v = std::getenv("HLM_ATTN_BWD");
  return v != nullptr && strcasecmp(v, "fused") == 0;
}

struct Attention : torch::autograd::Function<Attention> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                            int64_t window, double scale) {
    const std::vector<at::Tensor> res = fwd(q, k, v, window, scale, (int64_t)(uintptr_t)stream_of(q));
    ctx->save_for_backward({q, k, v, res[0], res[1]});
    ctx->saved_data["window"] = window;
    ctx->saved_data["scale"] = scale;
    return res[0];
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const int64_t window = ctx->saved_data["window"].toInt();
    const double scale = ctx->saved_data["scale"].toDouble();
    at::Tensor dout = grads[0];
    const at::Tensor none;
    if (needs_op({dout, s[0], s[1], s[2], s[3], s[4]}) || (s[0].size(3) == 64 && fused_backward_selected())) {
      const variable_list g =
          call_op("hip_attn_bwd", dout, s[0], s[1], s[2], s[3], s[4], window, scale);
      return {g[0], g[1], g[2], none, none};
    }
    const c10::Device dev = s[0].device();
    const c10::DeviceGuard guard(dev);
    const std::vector<int64_t> qsize = s[0].sizes().vec(), ksize = s[1].sizes().vec();
    const at::Tensor q = rows4(s[0], qsize, dev), k = rows4(s[1], ksize, dev), v = rows4(s[2], ksize, dev);
    const at::Tensor o = rows4(s[3], qsize, dev);
    dout = rows4(dout, qsize, dev);
    const int B = (int)qsize[0], T = (int)qsize[1], H = (int)qsize[2], Hkv = (int)ksize[2], D = (int)qsize[3];
    TORCH_CHECK(s[4].device() == dev && s[4].scalar_type() == at::kFloat && s[4].numel() == (int64_t)B * H * T,
                "a tensor of the backward does not match the forward's");
    const at::Tensor lse = s[4].contiguous();
    at::Tensor dq = at::empty(qsize, q.options()), dk = at::empty(ksize, q.options()), dv = at::empty(ksize, q.options());
    const auto f32 = q.options().dtype(at::kFloat);
    at::Tensor delta = at::empty({2 * (int64_t)B * H * T}, f32), part;
    const int64_t nbytes = hlm_attn_bwd_split_workspace_bytes(B, T, H, Hkv, D, (int)window);
    if (nbytes < 0) check((int)nbytes);
    if (nbytes > 0) part = at::empty({nbytes}, q.options().dtype(at::kByte));
    const Strides sq(q), sk(k), sv(v), so(o), sd(dout), sdq(dq), sdk(dk), sdv(dv);
    check(hlm_attn_bwd_split(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dout.data_ptr(),
                             lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), delta.data_ptr<float>(),
                             nbytes > 0 ? part.data_ptr() : nullptr, nbytes, B, T, H, Hkv, D, sq.s, sk.s, sv.s, so.s, sd.s,
                             sdq.s, sdk.s, sdv.s, (int)window, (float)scale, stream_of(q)));
    return {dq, dk, dv, none, none};
  }
};

// The differentiable attention call, or nothing where fwd takes nothing.
std::optional<at::Tensor> attn_train(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t window,
                                     double scale) {
  if (!plain(q) || !plain(k) || !plain(v) || !takes(q, k, v, window)) return std::nullopt;
  return Attention::apply(q, k, v, window, scale);
}

// A rotary table as (T, R) contiguous, 16-byte aligned rows in bf16 or fp32,
// or an undefined tensor.
at::Tensor rope_table(const at::Tensor& t, int64_t T) {
  if (!plain(t) || t.dim() == 0 || t.numel() != T * t.size(-1)) return {};
  if (t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kFloat) return {};
  at::Tensor r = t.detach().reshape({T, t.size(-1)}).contiguous();
  if (reinterpret_cast<uintptr_t>(r.data_ptr()) % 16 != 0) r = r.clone();
  return r;
}

bool heads4(const at::Tensor& t) { return plain(t) && t.dim() == 4 && t.scalar_type() == at::kBFloat16; }

struct QkNormRope : torch::autograd::Function<QkNormRope> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& cos,
                               const at::Tensor& sin, double eps) {
    const int64_t T = q.size(1), D = q.size(3);
    const at::Tensor c = rope_table(cos, T), s = rope_table(sin, T);
    at::Tensor qo = at::empty(q.sizes(), q.options()), ko = at::empty(k.sizes(), k.options());
    const Strides sq(q), sk(k);
    check(hlm_qk_norm_rope_fwd(q.data_ptr(), k.data_ptr(), c.data_ptr(), s.data_ptr(),
                               c.scalar_type() == at::kFloat ? HLM_TABLE_F32 : HLM_TABLE_BF16, qo.data_ptr(),
                               ko.data_ptr(), (int)q.size(0), (int)T, (int)q.size(2), (int)k.size(2), (int)D,
                               (int)c.size(1), sq.s, sk.s, (float)eps, stream_of(q)));
    ctx->save_for_backward({q, k, cos, sin});
    ctx->saved_data["eps"] = eps;
    return {qo, ko};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1];
    const double eps = ctx->saved_data["eps"].toDouble();
    const at::Tensor none;
    if (needs_op({grads[0], grads[1], saved[0], saved[1], saved[2], saved[3]})) {
      const variable_list g = call_op("hip_qk_norm_rope_backward", q, k, grads[0], grads[1], saved[2], saved[3], eps);
      return {g[0], g[1], none, none, none};
    }
    const c10::Device dev = q.device();
    const c10::DeviceGuard guard(dev);
    const std::vector<int64_t> qsize = q.sizes().vec(), ksize = k.sizes().vec();
    const int64_t T = q.size(1), D = q.size(3);
    const at::Tensor qr = rows4(q, qsize, dev), kr = rows4(k, ksize, dev);
    at::Tensor g[2];
    for (int i = 0; i < 2; ++i) {
      g[i] = grads[i];
      TORCH_CHECK(g[i].device() == dev && g[i].sizes() == at::IntArrayRef(i == 0 ? qsize : ksize),
                  "a gradient does not match the forward's output");
      if (g[i].scalar_type() != at::kBFloat16) g[i] = g[i].to(at::kBFloat16);
      g[i] = g[i].contiguous();
    }
    const at::Tensor c = rope_table(saved[2], T), s = rope_table(saved[3], T);
    TORCH_CHECK(c.defined() && s.defined() && c.scalar_type() == s.scalar_type() && c.sizes() == s.sizes() &&
                    c.device() == dev && s.device() == dev,
                "the rotary tables of the backward do not match the forward's");
    at::Tensor dq = at::empty(qsize, qr.options()), dk = at::empty(ksize, qr.options());
    const Strides sq(qr), sk(kr);
    check(hlm_qk_norm_rope_bwd(qr.data_ptr(), kr.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), c.data_ptr(),
                               s.data_ptr(), c.scalar_type() == at::kFloat ? HLM_TABLE_F32 : HLM_TABLE_BF16,
                               dq.data_ptr(), dk.data_ptr(), (int)qsize[0], (int)T, (int)qsize[2], (int)ksize[2], (int)D,
                               (int)c.size(1), sq.s, sk.s, (float)eps, stream_of(qr)));
    return {dq, dk, none, none, none};
  }
};

// The differentiable producer call, or nothing for inputs of the general path.
std::optional<std::tuple<at::Tensor, at::Tensor>> qk_norm_rope_train(const at::Tensor& q, const at::Tensor& k,
                                                                     const at::Tensor& cos, const at::Tensor& sin,
                                                                     double eps) {
  if (!heads4(q) || !heads4(k) || q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3))
    return std::nullopt;
  if (!kernel_ready(q) || !kernel_ready(k) || q.numel() > INT32_MAX || k.numel() > INT32_MAX) return std::nullopt;
  const at::Tensor c = rope_table(cos, q.size(1)), s = rope_table(sin, q.size(1));
  if (!c.defined() || !s.defined() || c.scalar_type() != s.scalar_type() || c.sizes() != s.sizes()) return std::nullopt;
  if (k.device() != q.device() || c.device() != q.device() || s.device() != q.device()) return std::nullopt;
  const c10::DeviceGuard guard(q.device());
  const variable_list out = QkNormRope::apply(q, k, cos, sin, eps);
  return std::make_tuple(out[0], out[1]);
}

// Contiguous 16-byte aligned bf16 rows.
at::Tensor rows2(at::Tensor t, at::IntArrayRef sizes, c10::Device device) {
  TORCH_CHECK(t.device() == device && t.sizes() == sizes, "a tensor of the backward does not match the forward's");
  if (t.scalar_type() != at::kBFloat16) t = t.to(at::kBFloat16);
  t = t.contiguous();
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone();
}

bool rows_ready(const at::Tensor& t) {
  return plain(t) && t.dim() >= 1 && t.scalar_type() == at::kBFloat16 && t.is_contiguous() &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct ResidualRmsNorm : torch::autograd::Function<ResidualRmsNorm> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& residual, const at::Tensor& branch, double eps) {
    const int64_t n = residual.size(-1);
    at::Tensor out = at::empty(residual.sizes(), residual.options()), normed = at::empty_like(out);
    check(hlm_residual_rms_norm_fwd(residual.data_ptr(), branch.data_ptr(), out.data_ptr(), normed.data_ptr(),
                                    n == 0 ? 0 : residual.numel() / n, (int)n, (float)eps, stream_of(residual)));
    ctx->save_for_backward({out});
    ctx->saved_data["eps"] = eps;
    return {out, normed};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::Tensor saved = ctx->get_saved_variables()[0];
    const double eps = ctx->saved_data["eps"].toDouble();
    if (needs_op({grads[0], grads[1], saved})) {
      const variable_list g =
          call_op("hip_residual_rms_norm_backward", saved, grads[0], grads[1], eps);
      return {g[0], g[0], at::Tensor()};
    }
    const c10::Device dev = saved.device();
    const c10::DeviceGuard guard(dev);
    const std::vector<int64_t> size = saved.sizes().vec();
    const int64_t n = size.back();
    const at::Tensor o = rows2(saved, size, dev), go = rows2(grads[0], size, dev), gn = rows2(grads[1], size, dev);
    at::Tensor g = at::empty(size, o.options());
    check(hlm_residual_rms_norm_bwd(o.data_ptr(), go.data_ptr(), gn.data_ptr(), g.data_ptr(), n == 0 ? 0 : o.numel() / n,
                                    (int)n, (float)eps, stream_of(o)));
    return {g, g, at::Tensor()};
  }
};

// The differentiable residual add + RMSNorm, or nothing for inputs of the
// general path.
std::optional<std::tuple<at::Tensor, at::Tensor>> residual_rms_norm_train(const at::Tensor& residual,
                                                                          const at::Tensor& branch, double eps) {
  if (!rows_ready(residual) || !rows_ready(branch) || residual.sizes() != branch.sizes() ||
      residual.device() != branch.device() || residual.size(-1) > INT32_MAX)
    return std::nullopt;
  const c10::DeviceGuard guard(residual.device());
  const variable_list out = ResidualRmsNorm::apply(residual, branch, eps);
  return std::make_tuple(out[0], out[1]);
}

}  // namespace

PYBIND11_MODULE(_torch_fwd, m) {
  m.doc() = "Host work of plain eager hip calls in C++: the no-grad forward and the differentiable calls.";
  m.def("fwd", &fwd, "fwd(q, k, v, window, scale, stream) -> [o, lse], or [] when the inputs need the general path");
  m.def("attn_train", &attn_train, "attn_train(q, k, v, window, scale) -> o, or None");
  m.def("qk_norm_rope_train", &qk_norm_rope_train, "qk_norm_rope_train(q, k, cos, sin, eps) -> (q, k), or None");
  m.def("residual_rms_norm_train", &residual_rms_norm_train,
        "residual_rms_norm_train(residual, branch, eps) -> (out, normed), or None");
}
