// Host path of the operators in native code: the allocations and the C ABI
// call (include/flash_spacetime.h) of one forward or one backward, on the
// operands in the form nearly every call gives them. What the Python layer
// (forward.py, backward.py) decides by some forty tensor calls and a 25-argument
// ctypes call is decided here in one: 63 -> 42 us a forward of one 187-token
// event (its kernel takes 16), 252 -> 154 us a forward and backward of 64 events
// of up to 192 tokens (its kernels then took 138, now 119).
//
// Both functions return None for anything but that form (unsupported shapes
// and dtypes, mixed devices, tensor subclasses, lengths that are not integers
// on the device, heads in groups, a call the library refuses): the caller then
// takes the Python path, which handles or rejects it. The library refuses
// before it launches a kernel; operands may have been converted by then. A
// call that failed otherwise (a launch error, a pending error of the device)
// raises: it is not run a second time. Nothing is kept between calls but the
// library's entry points.
#include <torch/extension.h>

#include <ATen/TensorSubclassLikeUtils.h>

#include <cmath>
#include <optional>
#include <stdexcept>
#include <string>

#include "../../include/flash_spacetime.h"

namespace {

namespace py = pybind11;
using at::Tensor;

struct Library {
  decltype(&fst_supported) supported = nullptr;
  decltype(&fst_forward_workspace_bytes) forward_workspace_bytes = nullptr;
  decltype(&fst_forward) forward = nullptr;
  decltype(&fst_backward_workspace_bytes) backward_workspace_bytes = nullptr;
  decltype(&fst_backward) backward = nullptr;
  decltype(&fst_last_error) last_error = nullptr;
} lib;

void bind_library(size_t supported, size_t fwd_ws, size_t fwd, size_t bwd_ws, size_t bwd, size_t last_error) {
  lib.supported = reinterpret_cast<decltype(lib.supported)>(supported);
  lib.forward_workspace_bytes = reinterpret_cast<decltype(lib.forward_workspace_bytes)>(fwd_ws);
  lib.forward = reinterpret_cast<decltype(lib.forward)>(fwd);
  lib.backward_workspace_bytes = reinterpret_cast<decltype(lib.backward_workspace_bytes)>(bwd_ws);
  lib.backward = reinterpret_cast<decltype(lib.backward)>(bwd);
  lib.last_error = reinterpret_cast<decltype(lib.last_error)>(last_error);
}

// Whether the library refused the call (a status it returns before any
// launch); any other failure raises with the library's message.
bool refused(int rc, const char* what) {
  if (rc == FST_EINVAL || rc == FST_EUNSUPPORTED) return true;
  if (rc != FST_OK) throw std::runtime_error(std::string(what) + ": " + lib.last_error());
  return false;
}

// A plain strided tensor on `dev`: no subclass, functorch wrapper, lazy
// conjugate or negation.
bool plain(const Tensor& t, const at::Device& dev) {
  return t.defined() && t.layout() == at::kStrided && t.device() == dev && !at::isTensorSubclassLike(t) &&
         !t.is_neg() && !t.is_conj();
}

// The heads-first view of dense [B, L, H, D] memory (forward.is_token_major).
bool token_major_view(const Tensor& t) { return !t.is_contiguous() && t.transpose(1, 2).is_contiguous(); }

bool width_ok(int64_t x) { return x == 16 || x == 32 || x == 48 || x == 64; }

void* data(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// Autograd is the caller's: its Function records the call.
struct NoGrad {
  at::AutoDispatchBelowADInplaceOrView below;
};

// Slot i of an interleaved [B, L, 3, H, D] (as [B, H, L, D]) or packed
// [T, 3, H, D] tensor.
Tensor slot(const Tensor& qkv, int64_t i, bool packed) {
  return packed ? qkv.select(1, i) : qkv.select(2, i).transpose(1, 2);
}

// q, k, v, or with k and v absent one contiguous interleaved tensor as q.
py::object forward_call(const Tensor& q_in, const std::optional<Tensor>& k_in, const std::optional<Tensor>& v_in,
                        const Tensor& feats, const Tensor& weight, const std::optional<Tensor>& bias,
                        const Tensor& lens, std::optional<double> scale, bool attn, bool act, bool packed,
                        int64_t stream) {
  const at::Device dev = q_in.device();
  const bool interleaved = !k_in.has_value();
  if (!lib.forward || !dev.is_cuda() || interleaved != !v_in.has_value()) return py::none();
  for (const Tensor* t : {&q_in, &feats, &weight, &lens})
    if (!plain(*t, dev)) return py::none();
  for (const auto* t : {&k_in, &v_in, &bias})
    if (t->has_value() && !plain(**t, dev)) return py::none();
  NoGrad guard;
  if (interleaved && (!q_in.is_contiguous() || q_in.dim() != (packed ? 4 : 5) || q_in.size(packed ? 1 : 2) != 3))
    return py::none();
  const Tensor q = interleaved ? slot(q_in, 0, packed) : q_in, k = interleaved ? slot(q_in, 1, packed) : *k_in,
               v = interleaved ? slot(q_in, 2, packed) : *v_in;
  const bool bf = q.scalar_type() == at::kBFloat16;
  if ((!bf && q.scalar_type() != at::kFloat) || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type())
    return py::none();
  if (q.dim() != (packed ? 3 : 4) || k.sizes() != q.sizes() || v.sizes() != q.sizes()) return py::none();
  const int64_t H = q.size(1), D = q.size(-1), L = packed ? 0 : q.size(2), T = packed ? q.size(0) : 0;
  const auto lt = lens.scalar_type();
  if (lens.dim() != 1 || (lt != at::kInt && lt != at::kLong)) return py::none();
  const int64_t B = packed ? lens.size(0) - 1 : q.size(0);
  if (B < 1 || (!packed && lens.size(0) != B) || H < 1 || (packed ? T : L) < 1) return py::none();
  if (packed ? feats.dim() != 2 || feats.size(0) != T
             : feats.dim() != 3 || feats.size(0) != B || feats.size(1) != L)
    return py::none();
  if (feats.size(-1) < 4 || !feats.is_floating_point()) return py::none();
  if (weight.dim() != 2 || weight.size(0) != D || !weight.is_floating_point()) return py::none();
  const int64_t C = weight.size(1);
  if (!width_ok(C) || !width_ok(D)) return py::none();
  if (bias.has_value() && (bias->dim() != 1 || bias->size(0) != D || !bias->is_floating_point())) return py::none();
  const double sc = scale.has_value() ? *scale : std::pow((double)D, -0.5);
  const int dtype = bf ? FST_BF16 : FST_F32;
  if (!lib.supported(dtype, (int)H, (int)D, (int)C)) return py::none();
  // Sizes the library's ints hold; a packed batch that could hold an event
  // past the 32-bit offsets is read back by the Python path.
  if (B > INT32_MAX / 16 || L > INT32_MAX / 16 || T > INT32_MAX / 16) return py::none();
  if (packed && T * H * (bf ? 2 : 4) * std::max(D * (interleaved ? 3 : 1), C) >= (int64_t)1 << 31) return py::none();

  c10::DeviceGuard on(dev);
  const bool tm = !packed && (interleaved || (token_major_view(q) && token_major_view(k) && token_major_view(v)));
  const int flags = (attn ? FST_ATTN_BIAS : 0) | (act ? FST_ACT_BIAS : 0) | (packed ? FST_PACKED : 0) |
                    (tm ? FST_TOKEN_MAJOR : 0) | (interleaved ? FST_QKV_INTERLEAVED : 0);
  const bool in_place = tm || interleaved;
  const Tensor qc = in_place ? q : q.contiguous(), kc = in_place ? k : k.contiguous(),
               vc = in_place ? v : v.contiguous();
  const Tensor pos4 = (feats.size(-1) == 4 ? feats : feats.narrow(-1, 0, 4)).to(at::kFloat).contiguous();
  const Tensor w32 = weight.detach().to(at::kFloat).contiguous();
  const Tensor b32 = bias.has_value() ? bias->detach().to(at::kFloat).contiguous() : Tensor();
  const Tensor len32 = lens.to(at::kInt).contiguous();
  const auto opt = q.options().requires_grad(false);
  Tensor out = !interleaved ? at::empty_like(qc)
               : packed     ? at::empty({T, H, D}, opt)
                            : at::empty({B, L, H, D}, opt).transpose(1, 2);
  const auto f32 = opt.dtype(at::kFloat);
  Tensor lse = packed ? at::empty({T, H}, f32)
               : tm   ? at::empty({B, L, H}, f32).transpose(1, 2)
                      : at::empty({B, H, L}, f32);
  const size_t bytes = lib.forward_workspace_bytes(dtype, flags, (int)B, (int)H, (int)L, (int)T, (int)D, (int)C);
  const Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 1)}, opt.dtype(at::kByte));
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = lib.forward(dtype, flags, (int)B, (int)H, (int)L, (int)T, (int)D, (int)C, data(qc), data(kc), data(vc),
                     static_cast<const float*>(data(pos4)), static_cast<const float*>(data(w32)),
                     static_cast<const float*>(data(b32)), static_cast<const int32_t*>(data(len32)), (float)sc,
                     data(out), static_cast<float*>(data(lse)), data(ws), bytes, reinterpret_cast<void*>(stream));
  }
  if (refused(rc, "flash_spacetime_forward")) return py::none();
  return py::make_tuple(out, lse, qc, kc, vc, pos4, w32, bias.has_value() ? py::cast(b32) : py::none(), len32,
                        py::make_tuple(dtype, flags, B, H, L, T, D, C), sc);
}

// dims as the forward returned them; q, k, v, or with k and v absent the
// interleaved tensor as q (its gradient is then one tensor of that layout).
// The tensors may have passed through the caller's saved-tensor hooks: their
// shapes and layouts are checked again before their addresses are used.
using Dims = std::tuple<int, int, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t>;
py::object backward_call(const Dims& dims, const Tensor& q_in, const std::optional<Tensor>& k_in,
                         const std::optional<Tensor>& v_in, const Tensor& pos4, const Tensor& w32,
                         const std::optional<Tensor>& b32, const Tensor& lens, const Tensor& lse,
                         const Tensor& grad_out, double scale, const std::optional<Tensor>& out, int64_t stream) {
  const at::Device dev = q_in.device();
  if (!lib.backward || !dev.is_cuda()) return py::none();
  for (const Tensor* t : {&q_in, &pos4, &w32, &lens, &lse, &grad_out})
    if (!plain(*t, dev)) return py::none();
  for (const auto* t : {&k_in, &v_in, &b32})
    if (t->has_value() && !plain(**t, dev)) return py::none();
  const auto [dtype, flags, B, H, L, T, D, C] = dims;
  const bool packed = flags & FST_PACKED, tm = flags & FST_TOKEN_MAJOR, inter = flags & FST_QKV_INTERLEAVED;
  if (inter == k_in.has_value() || inter == v_in.has_value()) return py::none();
  NoGrad guard;
  if (inter && (!q_in.is_contiguous() ||
                !(packed ? q_in.sizes() == at::IntArrayRef({T, 3, H, D}) : q_in.sizes() == at::IntArrayRef({B, L, 3, H, D}))))
    return py::none();
  const Tensor q = inter ? slot(q_in, 0, packed) : q_in, k = inter ? slot(q_in, 1, packed) : *k_in,
               v = inter ? slot(q_in, 2, packed) : *v_in;
  if (grad_out.sizes() != q.sizes()) return py::none();
  const auto st = dtype == FST_BF16 ? at::kBFloat16 : at::kFloat;
  if (packed ? q.dim() != 3 || q.size(0) != T : q.dim() != 4 || q.size(0) != B || q.size(2) != L) return py::none();
  if (q.size(1) != H || q.size(-1) != D || !lib.supported(dtype, (int)H, (int)D, (int)C)) return py::none();
  for (const Tensor* t : {&q, &k, &v}) {
    if (t->sizes() != q.sizes() || t->scalar_type() != st) return py::none();
    if (!inter && !(tm ? t->transpose(1, 2).is_contiguous() : t->is_contiguous())) return py::none();
  }
  if (lse.scalar_type() != at::kFloat ||
      !(packed ? lse.dim() == 2 && lse.size(0) == T && lse.size(1) == H && lse.is_contiguous()
               : lse.dim() == 3 && lse.size(0) == B && lse.size(1) == H && lse.size(2) == L &&
                     (tm ? lse.transpose(1, 2).is_contiguous() : lse.is_contiguous())))
    return py::none();
  if (pos4.scalar_type() != at::kFloat || !pos4.is_contiguous() || pos4.numel() != 4 * (packed ? T : B * L) ||
      lens.scalar_type() != at::kInt || !lens.is_contiguous() || lens.numel() != B + (packed ? 1 : 0) ||
      w32.scalar_type() != at::kFloat || !w32.is_contiguous() || w32.numel() != D * C ||
      (b32.has_value() && (b32->scalar_type() != at::kFloat || b32->numel() != D || !b32->is_contiguous())))
    return py::none();

  c10::DeviceGuard on(dev);
  // grad_out, and with it out, in the kernels' layout: [T, H, D], token-major
  // or heads-first dense.
  auto dense = [&, tm = tm, packed = packed](const Tensor& t) {
    return tm && !packed ? t.transpose(1, 2).is_contiguous() : t.is_contiguous();
  };
  Tensor go = grad_out.to(st);
  if (!dense(go)) {
    const auto opt = q.options().requires_grad(false);
    const Tensor d = tm && !packed ? at::empty({B, L, H, D}, opt).transpose(1, 2) : at::empty(q.sizes(), opt);
    go = d.copy_(go);
  }
  Tensor o;
  if (out.has_value() && plain(*out, dev) && out->sizes() == go.sizes() && out->scalar_type() == st && dense(*out))
    o = *out;
  Tensor grad, dq, dk, dv;
  if (inter) {
    grad = at::empty_like(q_in);
    dq = slot(grad, 0, packed), dk = slot(grad, 1, packed), dv = slot(grad, 2, packed);
  } else {
    dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    if (!dense(dq) || !dense(dk) || !dense(dv)) return py::none();
  }
  const auto f32 = w32.options().requires_grad(false);
  Tensor dw = at::empty({D, C}, f32);
  Tensor db = b32.has_value() ? at::empty({D}, f32) : Tensor();
  const size_t bytes = lib.backward_workspace_bytes(dtype, flags, (int)B, (int)H, (int)L, (int)T, (int)D, (int)C);
  const Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 1)}, f32.dtype(at::kByte));
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = lib.backward(
      dtype, flags, (int)B, (int)H, (int)L, (int)T, (int)D, (int)C, data(q), data(k), data(v),
      static_cast<const float*>(data(pos4)), static_cast<const float*>(data(w32)),
      b32.has_value() ? static_cast<const float*>(data(*b32)) : nullptr, static_cast<const int32_t*>(data(lens)),
      static_cast<const float*>(data(lse)), data(go), data(o), (float)scale, data(dq), data(dk), data(dv),
      static_cast<float*>(data(dw)), static_cast<float*>(data(db)), nullptr, data(ws), bytes,
      reinterpret_cast<void*>(stream));
  }
  if (refused(rc, "flash_spacetime_backward")) return py::none();
  return py::make_tuple(inter ? grad : dq, inter ? Tensor() : dk, inter ? Tensor() : dv, dw, b32.has_value() ? py::cast(db) : py::none());
}

// A failed allocation is the Python path's to report, with the exception type
// torch gives it there. Any other tensor error raises here.
template <typename F, typename... A>
py::object or_none(F f, const A&... args) {
  try {
    return f(args...);
  } catch (const c10::OutOfMemoryError&) {
    return py::none();
  }
}

py::object forward(const Tensor& q, const std::optional<Tensor>& k, const std::optional<Tensor>& v,
                   const Tensor& feats, const Tensor& weight, const std::optional<Tensor>& bias, const Tensor& lens,
                   std::optional<double> scale, bool attn, bool act, bool packed, int64_t stream) {
  return or_none(forward_call, q, k, v, feats, weight, bias, lens, scale, attn, act, packed, stream);
}

py::object backward(const Dims& dims, const Tensor& q, const std::optional<Tensor>& k, const std::optional<Tensor>& v,
                    const Tensor& pos4, const Tensor& w32, const std::optional<Tensor>& b32, const Tensor& lens,
                    const Tensor& lse, const Tensor& grad_out, double scale, const std::optional<Tensor>& out,
                    int64_t stream) {
  return or_none(backward_call, dims, q, k, v, pos4, w32, b32, lens, lse, grad_out, scale, out, stream);
}

}  // namespace

// build_id: the library this extension belongs to; torch_version: the torch it
// was compiled for (compared before bind_library gives it addresses).
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.attr("build_id") = FST_BUILD_ID;
  m.attr("torch_version") = FST_TORCH_VERSION;
  m.def("bind_library", &bind_library);
  m.def("forward", &forward);
  m.def("backward", &backward);
}
