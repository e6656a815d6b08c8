// fa_native.cpp — C++ autograd binding of libfa_gfx950.so for the public API's
// training path (host code only; built with g++ against PyTorch's headers).
//
// TritonAttention (the reference's torch.autograd.Function bridge,
// attention.py:673-771) runs its forward and backward in Python. At small
// shapes that costs more than the kernels: the Python Function's bookkeeping
// and the backward's trip through the autograd engine into Python take ~90 us
// per fwd+bwd on top of the op layer. This binding makes the same kernel
// launches from a C++ torch::autograd::Function, through fa_fwd_view and
// fa_bwd_view, with the same workspaces and on torch's current stream, so its
// results are identical bit for bit. forward() serves calls that need no
// gradient the same way (the op layer's flash_fwd, without the Python around
// it). Both serve positive scales and one head size, a multiple of 8, for q, k
// and v; attention.py keeps the Python path for the rest (negative or zero
// scales, other head sizes, forward-mode AD).
//
// The kernels read strided q, k, v and dO and head sizes below their width as
// they stand. Without gradients a model's transposed projections, slices of a fused
// projection and the filled part of a key/value cache are thus passed on without a
// copy (B1 Hq32 Hkv8 N3001 D128: the three copies took 34 us beside an 82 us forward;
// one query against a 3001-token part of a cache, 16 beside 23). operand() says
// which tensors qualify; the others are copied, as are k and v where their layouts
// differ (pair_up). With gradients q, k and v are copied once unless they are
// contiguous at a kernel's width (kept()), and dO is read as it stands where its
// layout is that of the q kept.
//
// The library's entry points come from the copy Python has already loaded
// (init() takes their addresses), so one libfa_gfx950.so serves both paths.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <stdexcept>
#include <string>

namespace {

using FwdView = int (*)(const void*, const void*, const void*, void*, void*, const int64_t*,
                        int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, float, int, void*,
                        int64_t, void*);
using BwdView = int (*)(const void*, const void*, const void*, const void*, const void*,
                        const void*, void*, void*, void*, void*, const int64_t*, int64_t, int64_t,
                        int64_t, int64_t, int64_t, int64_t, float, int, void*, int64_t, void*);
using WsBytes = int64_t (*)(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int);
using LastError = const char* (*)();

// Entry points; index 0 = fp16, 1 = bf16.
struct Entries {
  FwdView fwd[2] = {nullptr, nullptr};
  BwdView bwd[2] = {nullptr, nullptr};
  WsBytes fwd_ws_bytes = nullptr;
  WsBytes bwd_ws_bytes = nullptr;
  LastError last_error = nullptr;
};
Entries g;

bool ready() {
  return g.fwd[0] && g.fwd[1] && g.bwd[0] && g.bwd[1] && g.fwd_ws_bytes && g.bwd_ws_bytes &&
         g.last_error;
}

// The library's error as the Python binding words it (_lib.FlashAttentionError).
[[noreturn]] void fail(int64_t code) {
  throw std::runtime_error("libfa_gfx950 error " + std::to_string(code) + ": " +
                           std::string(g.last_error()));
}

void check(int64_t code) {
  if (code != 0) fail(code);
}

int elem_index(const at::Tensor& t) {
  if (t.scalar_type() == at::kHalf) return 0;
  if (t.scalar_type() == at::kBFloat16) return 1;
  throw std::invalid_argument("gfx950 attention: tensors must be float16 or bfloat16");
}

// The kernels move 128-bit vectors: a view whose data pointer is not 16-byte
// aligned is copied into a fresh allocation (as _ops._aligned does).
at::Tensor aligned(const at::Tensor& t) {
  const at::Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0
             ? c
             : c.clone(at::MemoryFormat::Contiguous);
}

// An input as the kernels read it: rows of consecutive columns, batches, heads and
// rows `stride` elements apart.
struct Operand {
  at::Tensor t;
  int64_t stride[3];
};

// Whether the kernels can read t [B, H, N, columns] as it stands: consecutive,
// 16-byte aligned rows that do not overlap, within 32-bit byte offsets of their
// head (the library's bounds, fa_capi.hip view_inputs). A dimension of one element
// has no stride to speak of.
bool readable(const at::Tensor& t) {
  if (t.is_neg() || t.stride(3) != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0)
    return false;
  for (int i = 0; i < 3; ++i)
    if (t.size(i) > 1 && t.stride(i) % 8 != 0) return false;
  if (t.size(1) > 1 && t.stride(1) >= (int64_t{1} << 35)) return false;
  const int64_t n = t.size(2), row = t.stride(2);
  return n == 1 || (row >= t.size(3) && row < (int64_t{1} << 30) &&
                    (n + 4096) * row * 2 < (int64_t{1} << 31));
}

Operand as_operand(const at::Tensor& t) {
  Operand o{t, {t.stride(0), t.stride(1), t.stride(2)}};
  // strides of one-element dimensions as a packed tensor has them
  if (t.size(2) == 1) o.stride[2] = t.size(3);
  if (t.size(1) == 1) o.stride[1] = t.size(2) * o.stride[2];
  if (t.size(0) == 1) o.stride[0] = t.size(1) * o.stride[1];
  return o;
}

Operand operand(const at::Tensor& t) {
  return as_operand(readable(t) ? t : aligned(t.resolve_neg()));
}

// Two operands that a kernel reads side by side need one layout: where theirs
// differ, the strided ones are copied.
void pair_up(Operand& a, Operand& b) {
  if (std::equal(a.stride, a.stride + 3, b.stride)) return;
  a = as_operand(aligned(a.t));
  b = as_operand(aligned(b.t));
}

// An input of a call with gradients, as it is saved for the backward: a contiguous one
// at a kernel width as it stands (a write before the backward then raises autograd's
// version error), any other one copied, so that the program may write its buffer (a
// fused projection, part of a key/value cache) before the backward. The copy is dense
// and keeps the order of the strides, so that q's copy pairs up with a dO of the same
// layout (a training step of B2 Hq32 Hkv8 N2048 D128 bf16 on projection views: 425 us;
// with the views themselves saved 401, with contiguous copies of all four 456).
at::Tensor kept(const at::Tensor& t) {
  const int64_t d = t.size(-1);
  if (t.is_contiguous() && (d == 32 || d == 64 || d == 128)) return t;
  return t.stride(-1) == 1 ? t.clone(at::MemoryFormat::Preserve)
                          : t.clone(at::MemoryFormat::Contiguous);
}

void* stream_of(const at::Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

// The uint8 workspace of `bytes` bytes (none for 0) from torch's caching allocator.
at::Tensor workspace(int64_t bytes, const at::Tensor& like) {
  if (bytes < 0) fail(bytes);
  return bytes > 0 ? at::empty({bytes}, like.options().dtype(at::kByte)) : at::Tensor();
}

struct Dims {
  int64_t B, Hq, Hkv, N, Nkv, D;
  // The kernel width that holds the head size (it sizes the workspaces).
  int64_t width() const { return D <= 32 ? 32 : D <= 64 ? 64 : 128; }
};

Dims dims_of(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4,
              "q, k, v must be 4-D [batch, heads, sequence, head_dim]");
  TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3),
              "k and v must have shape [B, Hkv, N_kv, D] matching q");
  TORCH_CHECK(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(),
              "q, k, v must share one dtype");
  TORCH_CHECK(q.is_cuda() && k.device() == q.device() && v.device() == q.device(),
              "q, k, v must be on one GPU");
  return {q.size(0), q.size(1), k.size(1), q.size(2), k.size(2), q.size(3)};
}

// The forward launch (the op layer's flash_fwd): O and the base-2 LSE of q, k, v
// (as the kernels read them) on the current stream of their device.
struct Forward {
  at::Tensor q, k, v, o, lse;
};

Forward run_forward(const at::Tensor& query, const at::Tensor& key, const at::Tensor& value,
                    bool causal, double scale) {
  const Dims d = dims_of(query, key, value);
  const int e = elem_index(query);
  c10::DeviceGuard guard(query.device());
  const Operand q = operand(query);
  Operand k = operand(key), v = operand(value);
  pair_up(k, v);
  Forward f{q.t, k.t, v.t, at::Tensor(), at::Tensor()};
  const int64_t strides[6] = {q.stride[0], q.stride[1], q.stride[2],
                              k.stride[0], k.stride[1], k.stride[2]};
  f.o = at::empty({d.B, d.Hq, d.N, d.D}, q.t.options());
  f.lse = at::empty({d.B, d.Hq, d.N}, q.t.options().dtype(at::kFloat));
  const int c = causal ? 1 : 0;
  const int64_t ws_bytes = g.fwd_ws_bytes(d.B, d.Hq, d.Hkv, d.N, d.Nkv, d.width(), c);
  const at::Tensor ws = workspace(ws_bytes, q.t);
  check(g.fwd[e](q.t.data_ptr(), k.t.data_ptr(), v.t.data_ptr(), f.o.data_ptr(), f.lse.data_ptr(),
                 strides, d.B, d.Hq, d.Hkv, d.N, d.Nkv, d.D, static_cast<float>(scale), c,
                 ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream_of(q.t)));
  return f;
}

class FlashAttention : public torch::autograd::Function<FlashAttention> {
 public:
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& query,
                            const at::Tensor& key, const at::Tensor& value, bool causal,
                            double scale) {
    Forward f = run_forward(kept(query), kept(key), kept(value), causal, scale);
    ctx->save_for_backward({f.q, f.k, f.v, f.o, f.lse});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    return f.o;
  }

  // The strides are read from the saved tensors as they come back (a saved-tensor
  // hook may return them laid out otherwise than they were packed).
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Dims d = dims_of(saved[0], saved[1], saved[2]);
    const int e = elem_index(saved[0]);
    c10::DeviceGuard guard(saved[0].device());
    Operand q = operand(saved[0]), k = operand(saved[1]), v = operand(saved[2]);
    Operand dO = operand(grads[0]);
    pair_up(k, v);
    pair_up(q, dO);
    const at::Tensor o = aligned(saved[3]), lse = aligned(saved[4]);
    const bool causal = ctx->saved_data["causal"].toBool();
    const float s = static_cast<float>(ctx->saved_data["scale"].toDouble());
    const int64_t strides[6] = {q.stride[0], q.stride[1], q.stride[2],
                                k.stride[0], k.stride[1], k.stride[2]};
    const int c = causal ? 1 : 0;
    const int64_t ws_bytes = g.bwd_ws_bytes(d.B, d.Hq, d.Hkv, d.N, d.Nkv, d.width(), c);
    const auto like = q.t.options();
    at::Tensor delta = at::empty({d.B, d.Hq, d.N}, like.dtype(at::kFloat));
    at::Tensor dq = at::empty({d.B, d.Hq, d.N, d.D}, like);
    at::Tensor dk = at::empty({d.B, d.Hkv, d.Nkv, d.D}, like);
    at::Tensor dv = at::empty({d.B, d.Hkv, d.Nkv, d.D}, like);
    const at::Tensor ws = workspace(ws_bytes, q.t);
    check(g.bwd[e](q.t.data_ptr(), k.t.data_ptr(), v.t.data_ptr(), o.data_ptr(),
                   dO.t.data_ptr(), lse.data_ptr(), delta.data_ptr(), dq.data_ptr(),
                   dk.data_ptr(), dv.data_ptr(), strides, d.B, d.Hq, d.Hkv, d.N, d.Nkv, d.D, s, c,
                   ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream_of(q.t)));
    return {dq, dk, dv, at::Tensor(), at::Tensor()};
  }
};

// O = attention(query, key, value) with the library's kernels, differentiable
// in query, key and value (see the file comment for the cases served).
at::Tensor attention(const at::Tensor& query, const at::Tensor& key, const at::Tensor& value,
                     bool causal, double scale) {
  if (!ready()) throw std::runtime_error("gfx950 attention: init() has not run");
  return FlashAttention::apply(query, key, value, causal, scale);
}

// O without autograd (inference: no input needs a gradient).
at::Tensor forward_only(const at::Tensor& query, const at::Tensor& key, const at::Tensor& value,
                        bool causal, double scale) {
  if (!ready()) throw std::runtime_error("gfx950 attention: init() has not run");
  return run_forward(query, key, value, causal, scale).o;
}

// The softmax scale of a public call that passes every check of attention.py
// (arguments, _validate_inputs, _decide_rules but the device's architecture,
// _kernel_scale) well inside its bounds, at one head size that is a multiple of 8;
// 0.0 for any other call, which attention.py then checks itself, one rule at a time, to
// word its error or choose its path. In Python the checks of a small call took as
// long as its forward launch (11-12 us for the two, 4.7 for the launch).
double plain_scale(py::handle query, py::handle key, py::handle value, py::handle is_causal,
                   py::handle scale, py::handle enable_gqa) {
  if (!THPVariable_CheckExact(query.ptr()) || !THPVariable_CheckExact(key.ptr()) ||
      !THPVariable_CheckExact(value.ptr()) || !PyBool_Check(is_causal.ptr()) ||
      !PyBool_Check(enable_gqa.ptr()))
    return 0.0;
  const at::Tensor& q = THPVariable_Unpack(query.ptr());
  const at::Tensor& k = THPVariable_Unpack(key.ptr());
  const at::Tensor& v = THPVariable_Unpack(value.ptr());
  const at::ScalarType dtype = q.scalar_type();
  if ((dtype != at::kHalf && dtype != at::kBFloat16) || k.scalar_type() != dtype ||
      v.scalar_type() != dtype || !q.is_cuda() || k.device() != q.device() ||
      v.device() != q.device() || q.dim() != 4 || k.dim() != 4 || v.sizes() != k.sizes())
    return 0.0;
  const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2), D = q.size(3);
  const int64_t Hkv = k.size(1), Nkv = k.size(2);
  constexpr int64_t kMany = int64_t{1} << 20;
  const auto within = [](int64_t n, int64_t most) { return n >= 1 && n <= most; };
  if (!within(B, kMany) || !within(Hq, kMany) || !within(Hkv, kMany) || !within(B * Hq, kMany) ||
      !within(N, kMany) || !within(Nkv, kMany) || !within(D, 128) || D % 8 != 0 ||
      k.size(0) != B || k.size(3) != D || Hq % Hkv != 0 ||
      (Hq != Hkv && enable_gqa.ptr() != Py_True))
    return 0.0;
  double s = 0.0;
  if (scale.is_none()) s = std::pow(static_cast<double>(D), -0.5);
  else if (PyFloat_CheckExact(scale.ptr())) s = PyFloat_AS_DOUBLE(scale.ptr());
  return s >= 1e-30 && s <= 1e30 ? s : 0.0;
}

// Takes the entry points' addresses: fa_fwd_view, fa_fwd_view_bf16, fa_bwd_view,
// fa_bwd_view_bf16, fa_fwd_workspace_bytes, fa_bwd_workspace_bytes, fa_last_error.
void init(int64_t fwd, int64_t fwd_bf16, int64_t bwd, int64_t bwd_bf16, int64_t fwd_ws_bytes,
          int64_t bwd_ws_bytes, int64_t last_error) {
  auto fn = [](int64_t a) { return reinterpret_cast<void*>(static_cast<uintptr_t>(a)); };
  Entries e;
  e.fwd[0] = reinterpret_cast<FwdView>(fn(fwd));
  e.fwd[1] = reinterpret_cast<FwdView>(fn(fwd_bf16));
  e.bwd[0] = reinterpret_cast<BwdView>(fn(bwd));
  e.bwd[1] = reinterpret_cast<BwdView>(fn(bwd_bf16));
  e.fwd_ws_bytes = reinterpret_cast<WsBytes>(fn(fwd_ws_bytes));
  e.bwd_ws_bytes = reinterpret_cast<WsBytes>(fn(bwd_ws_bytes));
  e.last_error = reinterpret_cast<LastError>(fn(last_error));
  g = e;
  if (!ready()) throw std::invalid_argument("gfx950 attention: a null entry point was passed");
}

}  // namespace

PYBIND11_MODULE(_fa_native, m) {
  m.doc() = "C++ autograd binding of libfa_gfx950.so (fa_fwd_view and fa_bwd_view)";
  m.def("init", &init);
  m.def("ready", &ready);
  m.def("attention", &attention);
  m.def("forward", &forward_only);
  m.def("plain_scale", &plain_scale);
}
