// The torch operators of chronicals_hip over the C ABI of libchronicals_cce
// (include/chronicals_cce.h): operand checks, output and workspace allocation,
// the current stream and one C call each.  In C++ because the same steps in
// Python take longer than the kernels of a small call: 16 rows of fp32 logits,
// V 151936, forward and backward (43 us of kernels) took 179 us with Python
// operators over ctypes and take 87 us with these; 64 rows of d 896 against
// V 32000 went from 222 to 143 us.
//
// ops.py defines the schemas and the fake (meta) implementations; the kernels
// are registered here.  The C functions come from the library that the Python
// loader opens (chronicals_torch_bind), so that CHRONICALS_CCE_LIB and the
// loader's checks hold for both.  The first call of an operator asks for it, and
// a failing call raises what the package's Python code raises: both through two
// Python callables that ops.py hands over (chronicals_torch_hooks).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/library.h>

#include <atomic>

#include "../../include/chronicals_cce.h"

namespace {

using at::Tensor;
using std::optional;

struct Api {
  decltype(&cce_last_error) last_error;
  decltype(&cce_forward_workspace_bytes) forward_workspace_bytes;
  decltype(&cce_backward_workspace_bytes) backward_workspace_bytes;
  decltype(&cce_forward) forward;
  decltype(&cce_backward) backward;
  decltype(&cce_logits_forward_workspace_bytes) logits_forward_workspace_bytes;
  decltype(&cce_logits_forward) logits_forward;
  decltype(&cce_logits_backward) logits_backward;
  decltype(&cce_logits_forward_backward) logits_forward_backward;
};

Api g_api;
std::atomic<bool> g_bound{false};

PyObject* g_load = nullptr;   // load(): opens the library and binds it here, or raises
PyObject* g_check = nullptr;  // check(rc): raises for a failing rc, with cce_last_error()'s text

// Calls a hook with its argument, if any; what it raises goes on as a Python
// exception.  Operators run without the interpreter's lock.
void call_hook(PyObject* hook, const long* arg) {
  TORCH_CHECK(hook != nullptr, "chronicals_amd.ops is not imported");
  struct Gil {
    PyGILState_STATE state = PyGILState_Ensure();
    ~Gil() { PyGILState_Release(state); }
  } gil;
  PyObject* const res = arg ? PyObject_CallFunction(hook, "l", *arg) : PyObject_CallObject(hook, nullptr);
  if (!res) {
    python_error e;
    e.persist();
    throw e;
  }
  Py_DECREF(res);
}

const Api& api() {
  if (!g_bound.load(std::memory_order_acquire)) call_hook(g_load, nullptr);
  TORCH_CHECK(g_bound.load(std::memory_order_acquire), "libchronicals_cce.so is not bound");
  return g_api;
}

// cce_last_error() is the calling thread's, and the hook runs in this thread.
void check(const Api& a, int rc) {
  if (rc == CCE_OK) return;
  const long code = rc;
  call_hook(g_check, &code);
  TORCH_CHECK(false, "libchronicals_cce error ", rc, ": ", a.last_error());
}

void* stream(const at::Device& device) {
  return c10::hip::getCurrentHIPStream(device.index()).stream();
}

// The kernels need 16-byte aligned rows: a view at an unaligned storage offset
// is copied to fresh storage.
Tensor aligned(const Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone();
}

bool is_label(const Tensor& t) { return t.scalar_type() == at::kLong || t.scalar_type() == at::kInt; }

void check_operands(const Tensor& hidden, const Tensor& weight, const Tensor& labels, const optional<Tensor>& bias) {
  TORCH_CHECK(hidden.scalar_type() == at::kBFloat16 && weight.scalar_type() == at::kBFloat16,
              "cce ops take bf16 hidden and weight, got ", hidden.scalar_type(), " and ", weight.scalar_type());
  TORCH_CHECK(hidden.dim() == 2 && weight.dim() == 2 && hidden.size(1) == weight.size(1),
              "cce ops take hidden [N, d] and weight [V, d], got ", hidden.sizes(), " and ", weight.sizes());
  TORCH_CHECK(labels.dim() == 1 && labels.size(0) == hidden.size(0) && is_label(labels),
              "cce ops take int64/int32 labels [N], got ", labels.scalar_type(), " ", labels.sizes());
  TORCH_CHECK(hidden.is_contiguous(), "hidden must be contiguous");
  TORCH_CHECK(weight.is_contiguous(), "weight must be contiguous");
  TORCH_CHECK(hidden.device() == weight.device() && hidden.device() == labels.device(),
              "hidden, weight and labels must be on the same device");
  if (bias.has_value())
    TORCH_CHECK(bias->scalar_type() == at::kFloat && bias->dim() == 1 && bias->size(0) == weight.size(0) &&
                    bias->is_contiguous() && bias->device() == hidden.device(),
                "bias must be a contiguous fp32 [V] tensor");
}

const float* bias_ptr(const optional<Tensor>& bias) {
  return bias.has_value() ? static_cast<const float*>(bias->data_ptr()) : nullptr;
}

// A per-row or scalar gradient as contiguous fp32.
Tensor grad_rows(const Tensor& g) { return g.detach().to(at::kFloat).reshape({-1}).contiguous(); }

std::tuple<Tensor, Tensor, Tensor, Tensor> cce_fwd(const Tensor& hidden_, const Tensor& weight_, const Tensor& labels_,
                                                   const optional<Tensor>& bias, int64_t ignore_index,
                                                   double label_smoothing, double z_loss_weight,
                                                   int64_t smoothing_form, int64_t reduction, int64_t lse_rows) {
  check_operands(hidden_, weight_, labels_, bias);
  const Api& a = api();
  const c10::DeviceGuard guard(hidden_.device());
  const Tensor hidden = aligned(hidden_), weight = aligned(weight_), labels = labels_.contiguous();
  const int64_t N = hidden.size(0), d = hidden.size(1), V = weight.size(0);
  size_t bytes = 0;
  check(a, a.forward_workspace_bytes(N, d, V, (int)reduction, (int)lse_rows, &bytes));
  const auto f32 = hidden.options().dtype(at::kFloat);
  const Tensor ws = at::empty({(int64_t)bytes}, hidden.options().dtype(at::kByte));
  Tensor loss = at::empty({reduction == CCE_REDUCTION_NONE ? N : 1}, f32);
  Tensor lse = at::empty({N}, f32), target = at::empty({N}, f32);
  Tensor n_valid = at::empty({1}, hidden.options().dtype(at::kInt));
  check(a, a.forward(hidden.data_ptr(), weight.data_ptr(), labels.data_ptr(), labels.scalar_type() == at::kLong,
                     bias_ptr(bias), N, d, V, ignore_index, (float)label_smoothing, (float)z_loss_weight,
                     (int)smoothing_form, (int)reduction, (int)lse_rows, static_cast<float*>(loss.data_ptr()),
                     static_cast<float*>(lse.data_ptr()), static_cast<float*>(target.data_ptr()),
                     static_cast<int32_t*>(n_valid.data_ptr()), ws.data_ptr(), bytes, stream(hidden.device())));
  return {loss, lse, n_valid, target};
}

std::tuple<Tensor, Tensor, Tensor> cce_bwd(const Tensor& grad_out, const Tensor& hidden_, const Tensor& weight_,
                                           const Tensor& labels_, const Tensor& lse, const Tensor& n_valid,
                                           const optional<Tensor>& bias, int64_t ignore_index, double label_smoothing,
                                           double z_loss_weight, int64_t reduction, int64_t chunk_size, bool need_dh,
                                           bool need_dw, bool need_db, bool dh_f32, bool dw_f32) {
  check_operands(hidden_, weight_, labels_, bias);
  TORCH_CHECK(!need_db || bias.has_value(), "need_db requires a bias");
  const Api& a = api();
  const c10::DeviceGuard guard(hidden_.device());
  const Tensor hidden = aligned(hidden_), weight = aligned(weight_), labels = labels_.contiguous();
  const int64_t N = hidden.size(0), d = hidden.size(1), V = weight.size(0);
  const Tensor g = grad_rows(grad_out);
  const auto f32 = hidden.options().dtype(at::kFloat);
  auto empty = [&](bool need, at::IntArrayRef size, bool f) {
    return need ? at::empty(size, f ? f32 : hidden.options()) : at::empty({0}, f ? f32 : hidden.options());
  };
  Tensor dh = empty(need_dh, {N, d}, dh_f32), dw = empty(need_dw, {V, d}, dw_f32), db = empty(need_db, {V}, true);
  if (need_dh || need_dw || need_db) {
    const int hdt = dh_f32 ? CCE_DTYPE_F32 : CCE_DTYPE_BF16, wdt = dw_f32 ? CCE_DTYPE_F32 : CCE_DTYPE_BF16;
    size_t bytes = 0;
    check(a, a.backward_workspace_bytes(N, d, V, chunk_size, need_dh, hdt, need_dw, wdt, &bytes));
    const Tensor ws = at::empty({(int64_t)bytes}, hidden.options().dtype(at::kByte));
    check(a, a.backward(static_cast<const float*>(g.data_ptr()), hidden.data_ptr(), weight.data_ptr(),
                        labels.data_ptr(), labels.scalar_type() == at::kLong, bias_ptr(bias),
                        static_cast<const float*>(lse.data_ptr()), static_cast<const int32_t*>(n_valid.data_ptr()), N,
                        d, V, ignore_index, (float)label_smoothing, (float)z_loss_weight, (int)reduction, chunk_size,
                        need_dh ? dh.data_ptr() : nullptr, hdt, need_dw ? dw.data_ptr() : nullptr, wdt,
                        need_db ? static_cast<float*>(db.data_ptr()) : nullptr, ws.data_ptr(), bytes,
                        stream(hidden.device())));
  }
  return {dh, dw, db};
}

int logits_dtype(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return CCE_DTYPE_BF16;
    case at::kHalf: return CCE_DTYPE_F16;
    case at::kFloat: return CCE_DTYPE_F32;
    default: TORCH_CHECK(false, "logits dtype ", t.scalar_type(), " not supported (bf16, fp16, fp32)");
  }
}

void check_logits(const Tensor& logits, const Tensor& labels) {
  logits_dtype(logits);
  TORCH_CHECK(logits.dim() == 2 && (logits.size(1) <= 1 || logits.stride(1) == 1),
              "ce_logits ops take [N, V] logits with a contiguous last dimension, got shape ", logits.sizes(),
              " strides ", logits.strides());
  TORCH_CHECK(labels.dim() == 1 && labels.size(0) == logits.size(0) && is_label(labels),
              "ce_logits ops take int64/int32 labels [N], got ", labels.scalar_type(), " ", labels.sizes());
  TORCH_CHECK(labels.is_contiguous(), "labels must be contiguous");
  TORCH_CHECK(labels.device() == logits.device(), "logits and labels must be on the same device");
}

int64_t row_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

struct LogitsOut {
  Tensor ws, loss, lse, n_valid;
  size_t bytes = 0;
  LogitsOut(const Api& a, const Tensor& logits, int64_t reduction) {
    const int64_t N = logits.size(0), V = logits.size(1);
    check(a, a.logits_forward_workspace_bytes(N, V, (int)reduction, &bytes));
    const auto f32 = logits.options().dtype(at::kFloat);
    ws = at::empty({(int64_t)bytes}, logits.options().dtype(at::kByte));
    loss = at::empty({reduction == CCE_REDUCTION_NONE ? N : 1}, f32);
    lse = at::empty({N}, f32);
    n_valid = at::empty({1}, logits.options().dtype(at::kInt));
  }
};

std::tuple<Tensor, Tensor, Tensor> ce_logits_fwd(const Tensor& logits, const Tensor& labels, int64_t ignore_index,
                                                 double label_smoothing, double z_loss_weight, int64_t smoothing_form,
                                                 int64_t reduction) {
  check_logits(logits, labels);
  const Api& a = api();
  const c10::DeviceGuard guard(logits.device());
  LogitsOut o(a, logits, reduction);
  check(a, a.logits_forward(logits.data_ptr(), logits_dtype(logits), row_stride(logits), labels.data_ptr(),
                            labels.scalar_type() == at::kLong, logits.size(0), logits.size(1), ignore_index,
                            (float)label_smoothing, (float)z_loss_weight, (int)smoothing_form, (int)reduction,
                            static_cast<float*>(o.loss.data_ptr()), static_cast<float*>(o.lse.data_ptr()),
                            static_cast<int32_t*>(o.n_valid.data_ptr()), o.ws.data_ptr(), o.bytes,
                            stream(logits.device())));
  return {o.loss, o.lse, o.n_valid};
}

Tensor gradient_like(const Tensor& logits, bool f32_grad) {
  return at::empty(logits.sizes(), f32_grad ? logits.options().dtype(at::kFloat) : logits.options());
}

Tensor ce_logits_bwd(const Tensor& grad_out, const Tensor& logits, const Tensor& labels, const Tensor& lse,
                     const Tensor& n_valid, int64_t ignore_index, double label_smoothing, double z_loss_weight,
                     int64_t smoothing_form, int64_t reduction, bool f32_grad) {
  check_logits(logits, labels);
  const Api& a = api();
  const c10::DeviceGuard guard(logits.device());
  Tensor dx = gradient_like(logits, f32_grad);
  if (logits.size(0) == 0) return dx;
  const Tensor g = grad_rows(grad_out);
  check(a, a.logits_backward(static_cast<const float*>(g.data_ptr()), logits.data_ptr(), logits_dtype(logits),
                             row_stride(logits), labels.data_ptr(), labels.scalar_type() == at::kLong,
                             static_cast<const float*>(lse.data_ptr()),
                             static_cast<const int32_t*>(n_valid.data_ptr()), logits.size(0), logits.size(1),
                             ignore_index, (float)label_smoothing, (float)z_loss_weight, (int)smoothing_form,
                             (int)reduction, dx.data_ptr(), logits_dtype(dx), row_stride(dx),
                             stream(logits.device())));
  return dx;
}

std::tuple<Tensor, Tensor, Tensor, Tensor> ce_logits_fwd_bwd(const Tensor& logits, const Tensor& labels,
                                                             int64_t ignore_index, double label_smoothing,
                                                             double z_loss_weight, int64_t smoothing_form,
                                                             int64_t reduction, bool grad_mean, bool f32_grad) {
  check_logits(logits, labels);
  const Api& a = api();
  const c10::DeviceGuard guard(logits.device());
  LogitsOut o(a, logits, reduction);
  Tensor dx = gradient_like(logits, f32_grad);
  check(a, a.logits_forward_backward(
               logits.data_ptr(), logits_dtype(logits), row_stride(logits), labels.data_ptr(),
               labels.scalar_type() == at::kLong, logits.size(0), logits.size(1), ignore_index,
               (float)label_smoothing, (float)z_loss_weight, (int)smoothing_form, (int)reduction, grad_mean,
               static_cast<float*>(o.loss.data_ptr()), static_cast<float*>(o.lse.data_ptr()),
               static_cast<int32_t*>(o.n_valid.data_ptr()), dx.data_ptr(), logits_dtype(dx), row_stride(dx),
               o.ws.data_ptr(), o.bytes, stream(logits.device())));
  return {o.loss, o.lse, o.n_valid, dx};
}

}  // namespace

extern "C" {

// Takes the C functions from an open libchronicals_cce; 0 when it has them all.
int chronicals_torch_bind(void* handle) {
  Api a;
  bool ok = true;
  auto get = [&](auto& fn, const char* name) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(dlsym(handle, name));
    ok = ok && fn != nullptr;
  };
  get(a.last_error, "cce_last_error");
  get(a.forward_workspace_bytes, "cce_forward_workspace_bytes");
  get(a.backward_workspace_bytes, "cce_backward_workspace_bytes");
  get(a.forward, "cce_forward");
  get(a.backward, "cce_backward");
  get(a.logits_forward_workspace_bytes, "cce_logits_forward_workspace_bytes");
  get(a.logits_forward, "cce_logits_forward");
  get(a.logits_backward, "cce_logits_backward");
  get(a.logits_forward_backward, "cce_logits_forward_backward");
  if (!ok) return 1;
  if (!g_bound.load(std::memory_order_acquire)) {
    g_api = a;
    g_bound.store(true, std::memory_order_release);
  }
  return 0;
}

// The Python callables of api() and check(); called with the interpreter's lock.
void chronicals_torch_hooks(PyObject* load, PyObject* check) {
  Py_XINCREF(load);
  Py_XINCREF(check);
  Py_XSETREF(g_load, load);
  Py_XSETREF(g_check, check);
}

}  // extern "C"

// HIP tensors carry the CUDA dispatch key in torch.
TORCH_LIBRARY_IMPL(chronicals_hip, CUDA, m) {
  m.impl("cce_fwd", cce_fwd);
  m.impl("cce_bwd", cce_bwd);
  m.impl("ce_logits_fwd", ce_logits_fwd);
  m.impl("ce_logits_bwd", ce_logits_bwd);
  m.impl("ce_logits_fwd_bwd", ce_logits_fwd_bwd);
}

// The operators have no derivative of their own (the autograd functions call
// them): a backward through one raises.
TORCH_LIBRARY_IMPL(chronicals_hip, Autograd, m) {
  for (const char* op : {"cce_fwd", "cce_bwd", "ce_logits_fwd", "ce_logits_bwd", "ce_logits_fwd_bwd"})
    m.impl(op, torch::autograd::autogradNotImplementedFallback());
}
