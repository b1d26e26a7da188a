// The hot torch.library ops (mxf8::quant_rows, adaln_quant_rows, gemm_rowwise, lora_down,
// attn_quant_kv, attn_fwd_q) as native kernels over the C ABI of libmxf8.  Their schemas and
// fake kernels are declared in minimaxh3_amd/ops.py; the kernels here take the CUDA and
// AutogradCUDA entries of the dispatcher (the device type of a ROCm GPU), where they stand in
// for the Python kernels of the declarations.
//
// What this path costs is what a short call costs: a Python op body (dispatch through two
// Python kernels, checks, ctypes) took about 20 us per launch, more than most launches of a
// few hundred tokens run on the GPU.  On an MI355X host, one FP8Linear call (two launches)
// 42.5 -> 16.4 us, one short attention call (four launches) 60.6 -> 33.5 us.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/library.h>

#include <atomic>

#include "../../include/mxf8.h"

namespace {

using at::Tensor;
using std::optional;

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// A non-zero status of the C ABI raises minimaxh3_amd._native.NativeError with the library's
// message (of this thread).
void check(int rc, const char* what) {
  if (rc == 0) return;
  const PyGILState_STATE gil = PyGILState_Ensure();
  PyObject* mod = PyImport_ImportModule("minimaxh3_amd._native");
  PyObject* res = mod ? PyObject_CallMethod(mod, "check", "is", rc, what) : nullptr;
  Py_XDECREF(res);
  Py_XDECREF(mod);
  if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed (status %d)", what, rc);
  python_error err;
  err.persist();
  PyGILState_Release(gil);
  throw err;
}

// The kernels are built for gfx950 only (checked once per device).
void require_gfx950(const Tensor& t, const char* what) {
  constexpr int kMax = 64;
  static std::atomic<int> known[kMax];
  TORCH_CHECK_VALUE(t.is_cuda(), what, ": expected a GPU tensor");
  const int idx = t.get_device();
  int ok = idx < kMax ? known[idx].load(std::memory_order_relaxed) : 0;
  if (ok == 0) {
    hipDeviceProp_t p;
    const bool gfx950 =
        hipGetDeviceProperties(&p, idx) == hipSuccess && std::string(p.gcnArchName).substr(0, 6) == "gfx950" &&
        (p.gcnArchName[6] == 0 || p.gcnArchName[6] == ':');
    ok = gfx950 ? 1 : 2;
    if (idx < kMax) known[idx].store(ok, std::memory_order_relaxed);
  }
  TORCH_CHECK(ok == 1, "minimaxh3_amd kernels need a gfx950 (MI355X) device, got cuda:", idx);
}

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return MXF8_BF16;
    case at::kHalf: return MXF8_F16;
    case at::kFloat: return MXF8_F32;
    default: TORCH_CHECK_VALUE(false, "unsupported dtype ", t.scalar_type());
  }
}

void on_device(const Tensor& t, at::Device dev, const char* what, const char* name) {
  TORCH_CHECK_VALUE(t.device() == dev, what, name, " must be on ", dev, ", got ", t.device());
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dt) {
  return at::empty(sizes, like.options().dtype(dt));
}

constexpr auto kE4M3 = at::kFloat8_e4m3fn;

std::tuple<Tensor, Tensor> quant_rows(const Tensor& x_in) {
  require_gfx950(x_in, "quant_rows");
  TORCH_CHECK_INDEX(x_in.dim() >= 2, "quant_rows: expected x [M, K], got ", x_in.dim(), " dimensions");
  TORCH_CHECK_VALUE(x_in.dim() == 2, "quant_rows: expected x [M, K]");
  const Tensor x = x_in.stride(1) != 1 || x_in.stride(0) < x_in.size(1) ? x_in.contiguous() : x_in;
  const int64_t M = x.size(0), K = x.size(1);
  Tensor x8 = empty({M, K}, x, kE4M3), scale = empty({M, 1}, x, at::kFloat);
  if (M > 0) {
    const c10::DeviceGuard guard(x.device());
    check(mxf8_quant_rows(x.data_ptr(), dtype_code(x), M, K, std::max(x.stride(0), K),
                          static_cast<uint8_t*>(x8.data_ptr()), scale.data_ptr<float>(), stream_of(x)),
          "quant_rows");
  }
  return {x8, scale};
}

std::tuple<Tensor, Tensor, Tensor> adaln_quant_rows(const Tensor& x, const Tensor& shift_in, const Tensor& scale_in,
                                                    double eps, bool eager, bool want_y) {
  require_gfx950(x, "adaln_quant_rows");
  TORCH_CHECK_VALUE(x.dim() == 3 && shift_in.dim() == 2 && shift_in.size(0) == x.size(0) &&
                        shift_in.size(1) == x.size(2) && scale_in.sizes() == shift_in.sizes(),
                    "adaln_quant_rows: expected x [B, S, C] and shift, scale [B, C]");
  TORCH_CHECK_VALUE(x.scalar_type() == at::kBFloat16 && shift_in.scalar_type() == at::kBFloat16 &&
                        scale_in.scalar_type() == at::kBFloat16,
                    "adaln_quant_rows: bf16 tensors expected");
  on_device(shift_in, x.device(), "adaln_quant_rows: ", "shift");
  on_device(scale_in, x.device(), "adaln_quant_rows: ", "scale");
  const int64_t B = x.size(0), S = x.size(1), C = x.size(2), M = B * S;
  Tensor x2 = x.reshape({M, C}), shift = shift_in, scale = scale_in;
  if (x2.stride(1) != 1) x2 = x2.contiguous();
  // one row stride for both (expanded / strided operands are copied)
  if (shift.stride(1) != 1 || shift.stride(0) < C || shift.stride(0) % 8) shift = shift.contiguous();
  if (scale.stride(1) != 1 || scale.stride(0) != shift.stride(0)) {
    scale = scale.contiguous();
    if (scale.stride(0) != shift.stride(0)) shift = shift.contiguous();
  }
  Tensor x8 = empty({M, C}, x, kE4M3), sa = empty({M, 1}, x, at::kFloat);
  Tensor y = want_y ? empty({M, C}, x, at::kBFloat16) : empty({0}, x, at::kBFloat16);
  if (M > 0) {
    const c10::DeviceGuard guard(x.device());
    check(mxf8_adaln_quant_rows(x2.data_ptr(), M, C, x2.stride(0), S, shift.data_ptr(), scale.data_ptr(),
                                shift.stride(0), static_cast<float>(eps), eager, static_cast<uint8_t*>(x8.data_ptr()),
                                sa.data_ptr<float>(), want_y ? y.data_ptr() : nullptr, stream_of(x)),
          "adaln_quant_rows");
  }
  return {x8, sa, y};
}

Tensor gemm_rowwise(const Tensor& a8, const Tensor& w8, const Tensor& sa, const Tensor& sw,
                    const optional<Tensor>& bias, int64_t act, const optional<Tensor>& lora_t,
                    const optional<Tensor>& lora_b, double lora_scale) {
  const char* what = "gemm_rowwise: ";
  require_gfx950(a8, "gemm_rowwise");
  TORCH_CHECK_VALUE(a8.dim() == 2 && a8.scalar_type() == kE4M3 && w8.scalar_type() == kE4M3 && w8.dim() == 2 &&
                        w8.size(1) == a8.size(1),
                    what, "e4m3 a8 [M, K] and w8 [N, K] expected, got ", a8.scalar_type(), " ", a8.sizes(), " and ",
                    w8.scalar_type(), " ", w8.sizes());
  const int64_t M = a8.size(0), K = a8.size(1), N = w8.size(0);
  TORCH_CHECK_VALUE(a8.is_contiguous() && w8.is_contiguous(), what, "a8 and w8 must be contiguous");
  TORCH_CHECK_VALUE(sa.scalar_type() == at::kFloat && sa.numel() == M && sw.scalar_type() == at::kFloat &&
                        sw.numel() == N,
                    what, "fp32 scales of ", M, " rows and ", N, " channels expected");
  TORCH_CHECK_VALUE(sa.is_contiguous() && sw.is_contiguous(), what, "scales must be contiguous");
  TORCH_CHECK_VALUE(!bias || (bias->scalar_type() == at::kBFloat16 && bias->numel() == N && bias->is_contiguous()),
                    what, "bias must be ", N, " contiguous bf16 values");
  TORCH_CHECK_VALUE(!lora_t || (lora_b && lora_t->dim() == 2 && lora_t->size(0) == M && lora_b->dim() == 2 &&
                                lora_b->size(0) == N && lora_b->size(1) == lora_t->size(1) &&
                                lora_t->scalar_type() == at::kBFloat16 && lora_b->scalar_type() == at::kBFloat16 &&
                                lora_t->is_contiguous() && lora_b->is_contiguous()),
                    what, "LoRA operands t [M, r] and B [N, r] (contiguous bf16) expected");
  const at::Device dev = a8.device();
  on_device(w8, dev, what, "w8");
  on_device(sa, dev, what, "sa");
  on_device(sw, dev, what, "sw");
  if (bias) on_device(*bias, dev, what, "bias");
  if (lora_t) on_device(*lora_t, dev, what, "lora_t");
  if (lora_b) on_device(*lora_b, dev, what, "lora_b");
  Tensor out = empty({M, N}, a8, at::kBFloat16);
  if (M == 0 || N == 0) return out;
  const c10::DeviceGuard guard(dev);
  check(mxf8_gemm_rowwise(static_cast<const uint8_t*>(a8.data_ptr()), static_cast<const uint8_t*>(w8.data_ptr()),
                          sa.data_ptr<float>(), sw.data_ptr<float>(), bias ? bias->data_ptr() : nullptr,
                          static_cast<int>(act), lora_t ? lora_t->data_ptr() : nullptr,
                          lora_b ? lora_b->data_ptr() : nullptr, lora_t ? lora_t->size(1) : 0,
                          static_cast<float>(lora_scale), out.data_ptr(), M, N, K, N, stream_of(a8)),
        "gemm_rowwise");
  return out;
}

Tensor lora_down(const Tensor& x_in, const Tensor& a_in) {
  require_gfx950(x_in, "lora_down");
  TORCH_CHECK_INDEX(x_in.dim() >= 2, "lora_down: expected x [M, K], got ", x_in.dim(), " dimensions");
  // (the kernel reads both as bf16 and addresses A by x's K)
  TORCH_CHECK_VALUE(x_in.dim() == 2 && a_in.dim() == 2 && a_in.size(1) == x_in.size(1) &&
                        x_in.scalar_type() == at::kBFloat16 && a_in.scalar_type() == at::kBFloat16,
                    "lora_down: bf16 x [M, K] and A [r, K] expected, got ", x_in.scalar_type(), " ", x_in.sizes(),
                    " and ", a_in.scalar_type(), " ", a_in.sizes());
  on_device(a_in, x_in.device(), "lora_down: ", "a");
  const Tensor x = x_in.stride(1) != 1 ? x_in.contiguous() : x_in, a = a_in.contiguous();
  const int64_t M = x.size(0), K = x.size(1), r = a.size(0);
  Tensor t = empty({M, r}, x, at::kBFloat16);
  if (M > 0) {
    const c10::DeviceGuard guard(x.device());
    check(mxf8_lora_down(x.data_ptr(), x.stride(0), a.data_ptr(), t.data_ptr(), M, K, r, stream_of(x)), "lora_down");
  }
  return t;
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> attn_quant_kv(const Tensor& k, const Tensor& v) {
  require_gfx950(k, "attn_quant_kv");
  TORCH_CHECK_VALUE(k.dim() == 4 && k.sizes() == v.sizes() && k.scalar_type() == v.scalar_type() &&
                        k.device() == v.device(),
                    "attn_quant_kv: k and v must have one shape, dtype and device");
  const int64_t B = k.size(0), H = k.size(1), S = k.size(2), D = k.size(3), nk = cdiv(S, 128);
  Tensor k8 = empty({B, H, nk * 128, D}, k, kE4M3), sk = empty({B, H, nk}, k, at::kFloat);
  Tensor v8t = empty({B, H, D, nk * 128}, k, kE4M3), sv = empty({B, H, D}, k, at::kFloat);
  Tensor mean = empty({B, H, D}, k, at::kFloat);
  Tensor ws = empty({std::max<int64_t>(mxf8_attn_kv_workspace_bytes(B, H, S, D), 16)}, k, at::kByte);
  const c10::DeviceGuard guard(k.device());
  check(mxf8_attn_quant_kv(k.data_ptr(), k.strides().data(), v.data_ptr(), v.strides().data(), dtype_code(k), B, H, S,
                           D, static_cast<uint8_t*>(k8.data_ptr()), sk.data_ptr<float>(),
                           static_cast<uint8_t*>(v8t.data_ptr()), sv.data_ptr<float>(), mean.data_ptr<float>(),
                           ws.data_ptr(), stream_of(k)),
        "attn_quant_kv");
  return {k8, sk, v8t, sv, mean};
}

// The K/V codes must have exactly the layout attn_quant_kv gives for Sk keys (the kernels
// address them through Sk alone).
void check_codes(const Tensor& t, at::IntArrayRef shape, at::ScalarType dt, const char* name, int64_t Sk,
                 at::Device dev) {
  TORCH_CHECK_VALUE(t.sizes() == shape && t.scalar_type() == dt && t.is_contiguous(), "attn_fwd_q: ", name,
                    " must be a contiguous ", dt, " tensor of shape ", shape, " for Sk=", Sk, ", got ",
                    t.scalar_type(), " ", t.sizes());
  on_device(t, dev, "attn_fwd_q: ", name);
}

// key_mask (bool) / key_bias (fp32) as one row of Sk values per batch item.
Tensor key_operand(const Tensor& t_in, at::ScalarType dt, const char* name, int64_t B, int64_t Sk, at::Device dev) {
  on_device(t_in, dev, "", name);
  Tensor t = t_in.to(dt);
  if (t.numel() == B * Sk)
    t = t.reshape({B, Sk});
  else if (t.numel() == Sk)
    t = t.reshape({1, Sk}).expand({B, Sk});
  else
    TORCH_CHECK_VALUE(false, name, " must hold B*Sk = ", B * Sk, " (or Sk = ", Sk, ") values, got shape ", t.sizes());
  return t.contiguous();
}

// As ops.attn_fwd_q_supported, for a 4-d q.
bool fused_q_layout(const Tensor& q) {
  return (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) && q.stride(3) == 1 &&
         q.stride(0) % 8 == 0 && q.stride(1) % 8 == 0 && q.stride(2) % 8 == 0;
}

Tensor attn_fwd_q(const Tensor& q, double c, const Tensor& k8, const Tensor& v8t, const Tensor& sk, const Tensor& sv,
                  const optional<Tensor>& key_mask, const optional<Tensor>& key_bias, double repair_tau, int64_t Sk,
                  int64_t kv_mode) {
  require_gfx950(q, "attn_fwd_q");
  TORCH_CHECK_VALUE(q.dim() == 4 && fused_q_layout(q),
                    "attn_fwd_q: q must be bf16/fp16 with unit channel stride, other strides multiples of 8 and "
                    "16-byte alignment");
  if (reinterpret_cast<uintptr_t>(q.data_ptr()) % 16) {
    // a view that starts off a 16-byte boundary: the two launches give the same bits
    static const auto quant_q = c10::Dispatcher::singleton()
                                    .findSchemaOrThrow("mxf8::attn_quant_q", "")
                                    .typed<std::tuple<Tensor, Tensor>(const Tensor&, double)>();
    static const auto fwd =
        c10::Dispatcher::singleton()
            .findSchemaOrThrow("mxf8::attn_fwd", "")
            .typed<Tensor(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                          const optional<Tensor>&, const optional<Tensor>&, double, const Tensor&, int64_t, int64_t)>();
    const auto [q8, sq] = quant_q.call(q, c);
    return fwd.call(q8, k8, v8t, sq, sk, sv, key_mask, key_bias, repair_tau, q, Sk, kv_mode);
  }
  const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Skp = cdiv(Sk, 128) * 128;
  const at::Device dev = q.device();
  check_codes(k8, {B, H, Skp, D}, kE4M3, "k8", Sk, dev);
  check_codes(v8t, {B, H, D, Skp}, kE4M3, "v8t", Sk, dev);
  check_codes(sk, {B, H, Skp / 128}, at::kFloat, "sk", Sk, dev);
  check_codes(sv, {B, H, D}, at::kFloat, "sv", Sk, dev);
  Tensor out = at::empty_like(q), km, kb;
  if (key_mask) km = key_operand(*key_mask, at::kBool, "key_mask", B, Sk, dev);
  if (key_bias) kb = key_operand(*key_bias, at::kFloat, "key_bias", B, Sk, dev);
  const c10::DeviceGuard guard(dev);
  check(mxf8_attn_fwd_q(q.data_ptr(), q.strides().data(), static_cast<float>(c),
                        static_cast<const uint8_t*>(k8.data_ptr()), static_cast<const uint8_t*>(v8t.data_ptr()),
                        sk.data_ptr<float>(), sv.data_ptr<float>(),
                        km.defined() ? static_cast<const uint8_t*>(km.data_ptr()) : nullptr,
                        kb.defined() ? kb.data_ptr<float>() : nullptr, static_cast<float>(repair_tau), nullptr,
                        out.data_ptr(), dtype_code(out), out.strides().data(), B, H, Sq, Sk, D,
                        static_cast<int>(kv_mode), stream_of(q)),
        "attn_fwd_q");
  return out;
}

// The ops have no derivative.  With grad mode on, an output of an input that requires grad
// requires grad and its backward raises; otherwise the call goes on below autograd (as the
// Python declarations' autograd kernel does; forward-mode tangents end here).
void no_derivative(const c10::OperatorHandle& op, c10::DispatchKeySet ks, torch::jit::Stack* stack) {
  const size_t nargs = op.schema().arguments().size();
  torch::autograd::edge_list edges;
  if (at::GradMode::is_enabled()) {
    bool any = false;
    for (size_t i = 0; i < nargs; ++i) {
      const c10::IValue& v = torch::jit::peek(*stack, i, nargs);
      any = any || (v.isTensor() && v.toTensor().defined() && v.toTensor().requires_grad());
    }
    if (any) {
      for (size_t i = 0; i < nargs; ++i) {
        const c10::IValue& v = torch::jit::peek(*stack, i, nargs);
        if (v.isTensor() && v.toTensor().defined() && v.toTensor().requires_grad())
          edges.push_back(torch::autograd::impl::gradient_edge(v.toTensor()));
      }
    }
  }
  {
    const at::AutoDispatchBelowAutograd guard;
    op.redispatchBoxed(ks & c10::after_autograd_keyset, stack);
  }
  if (edges.empty()) return;
  const std::string name = op.schema().name().substr(6);  // without "mxf8::"
  const auto node = std::make_shared<torch::autograd::Error>(
      "Trying to backward through mxf8." + name + ".default but no autograd formula was registered. Please use "
      "register_autograd to add one.", std::move(edges));
  const size_t nret = op.schema().returns().size();
  for (size_t i = 0; i < nret; ++i)
    torch::autograd::set_history(torch::jit::peek(*stack, i, nret).toTensor(), node);
}

}  // namespace

TORCH_LIBRARY_IMPL(mxf8, CUDA, m) {
  m.impl("quant_rows", &quant_rows);
  m.impl("adaln_quant_rows", &adaln_quant_rows);
  m.impl("gemm_rowwise", &gemm_rowwise);
  m.impl("lora_down", &lora_down);
  m.impl("attn_quant_kv", &attn_quant_kv);
  m.impl("attn_fwd_q", &attn_fwd_q);
}

TORCH_LIBRARY_IMPL(mxf8, AutogradCUDA, m) {
  for (const char* op : {"quant_rows", "adaln_quant_rows", "gemm_rowwise", "lora_down", "attn_quant_kv", "attn_fwd_q"})
    m.impl(op, torch::CppFunction::makeFromBoxedFunction<&no_derivative>());
}
