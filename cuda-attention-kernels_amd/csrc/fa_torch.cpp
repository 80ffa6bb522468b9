// Native dispatcher kernels of the custom op fused_attn::attention for GPU tensors.
//
// The op is defined in Python (fused_attn/ops.py), whose kernel checks, prepares and launches a call through
// ctypes: 20-27 us of host time, more than the GPU needs for a small call.  The kernels here take the calls
// that need no preparation (operands the HIP kernels read as they are, no backend forced by the environment, a
// device the Python side has found supported) and launch them in 6-8 us; every other call, errors included,
// goes on to the Python kernels, which stay the one place that says what is accepted and how it fails.
//
// The choice of kernel and partitions repeats ops._hip_kernel_for and ops.default_split_len
// (fa_torch_route lets a test compare the two).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>

#include "../../include/fused_attn_hip.h"

namespace {

// C ABI of the HIP library, set once by fa_torch_bind (ctypes has loaded the library, maybe from a path the
// user named), and the devices the Python side has found supported.
struct Abi {
  size_t (*fwd_workspace_bytes)(const fa_fwd_params*);
  fa_status (*fwd_ws)(const fa_fwd_params*, void*, size_t, void*);
  size_t (*splitk_workspace_bytes)(int32_t, int32_t, int32_t, int32_t, int32_t);
  fa_status (*splitk)(const fa_fwd_params*, int32_t, void*, size_t, void*);
  const char* (*last_error)();
};
Abi g_abi{};
std::atomic<uint64_t> g_devices{0};

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool is_short_decode(int64_t b, int64_t hq, int64_t hkv, int64_t nq, int64_t nk, int64_t d) {
  const int64_t group = hq / hkv, heads = b * hq;
  if (nq == 0 || group * nq > 32 || nq > 8) return false;
  if (heads <= 64) return d != 256 && (group > 1 || nq <= 4) && nk >= (d == 64 ? 641 : 512);
  const bool many = heads > (d == 256 ? 256 : 512);
  if (group < 4) {
    if (group == 1 || nq > 4) return false;
    if (nq > 2) return nk >= 1600;
    if (many) return nk >= (d == 64 ? 384 : 192);
    return nk >= (d == 64 ? 1000 : d == 128 ? 768 : 512);
  }
  if (nq > 4) return nk >= (d == 64 ? 1600 : 1280);
  if (many) return nk >= (d != 64 ? 192 : nq <= 2 ? 256 : 512);
  return nk >= (d != 64 ? 512 : nq <= 2 ? 641 : 1000);
}

// Keys per split-K partition, or 0 for the prefill kernel.
int64_t route(bool half, int64_t b, int64_t hq, int64_t hkv, int64_t nq, int64_t nk, int64_t d) {
  if (!half || !(d == 64 || d == 128 || d == 256)) return 0;
  if (!(nq <= 16 && nk >= 2048) && !is_short_decode(b, hq, hkv, nq, nk, d)) return 0;
  const int64_t items = std::max<int64_t>(1, b * hkv * ceil_div(hq / hkv * nq, 128));
  const int64_t parts = std::max<int64_t>(1, ceil_div(2048, items));
  const int64_t keys = ceil_div(ceil_div(std::max<int64_t>(nk, 1), parts), 64) * 64;
  return std::min<int64_t>(std::max<int64_t>(keys, 128), 4096);
}

// The kernels read t as it is: unit stride along D, 16-byte aligned rows, token strides below 16 MiB.
bool readable(const at::Tensor& t) {
  if (t.stride(3) != 1 || reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 != 0) return false;
  for (int i = 0; i < 3; ++i) {
    if (t.size(i) > 1 && t.stride(i) % 8 != 0) return false;
  }
  return t.size(2) <= 1 || t.stride(2) * (int64_t)t.element_size() < (int64_t{1} << 24);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return FA_DTYPE_F16;
    case at::kBFloat16: return FA_DTYPE_BF16;
    case at::kFloat: return FA_DTYPE_F32;
    default: return -1;
  }
}

// Whether the environment names a backend.  Read with the GIL held (torch calls kernels without it): os.environ sets
// variables under it, and a setenv beside this getenv may move the table it reads.
bool backend_forced() {
  const PyGILState_STATE gil = PyGILState_Ensure();
  const char* forced = std::getenv("FUSED_ATTN_BACKEND");
  const bool set = forced != nullptr && *forced != '\0';
  PyGILState_Release(gil);
  return set;
}

bool takes(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !q.is_cuda() || !k.is_cuda() || !v.is_cuda()) return false;
  const int dev = q.device().index();
  if (dev < 0 || dev >= 64 || !((g_devices.load(std::memory_order_acquire) >> dev) & 1)) return false;
  if (k.device() != q.device() || v.device() != q.device()) return false;
  if (q.layout() != at::kStrided || k.layout() != at::kStrided || v.layout() != at::kStrided) return false;
  if (dtype_code(q.scalar_type()) < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  if (!k.sizes().equals(v.sizes()) || k.size(3) != q.size(3) || (k.size(0) != q.size(0) && k.size(0) != 1)) return false;
  if (q.numel() == 0 || k.numel() == 0 || q.size(1) % k.size(1) != 0) return false;
  for (const at::Tensor* t : {&q, &k}) {
    for (const int64_t n : t->sizes()) {
      if (n > INT32_MAX) return false;
    }
  }
  if (!readable(q) || !readable(k) || !readable(v)) return false;
  return !backend_forced();
}

const c10::OperatorHandle& attention_op() {
  static const c10::OperatorHandle op = c10::Dispatcher::singleton().findSchemaOrThrow("fused_attn::attention", "");
  return op;
}

// The Python kernel registered under `key`.
at::Tensor call_python(c10::DispatchKey key, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal,
                       std::optional<double> scale) {
  torch::jit::Stack stack;
  torch::jit::push(stack, q, k, v, causal, scale);
  attention_op().callBoxedForDispatchKey(key, stack);
  return torch::jit::pop(stack).toTensor();
}

at::Tensor attention_gpu(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal,
                         std::optional<double> scale) {
  if (!takes(q, k, v)) return call_python(c10::DispatchKey::CompositeExplicitAutograd, q, k, v, causal, scale);
  const c10::DeviceGuard guard(q.device());
  at::Tensor o = at::empty(q.sizes(), q.options());
  fa_fwd_params p{};
  auto strides = [](const at::Tensor& t, int64_t& b, int64_t& h, int64_t& n) {
    b = t.size(0) > 1 ? t.stride(0) : 0;  // a dimension of size 1 is never stepped over
    h = t.size(1) > 1 ? t.stride(1) : 0;
    n = t.size(2) > 1 ? t.stride(2) : 0;
  };
  p.q = q.const_data_ptr();
  p.k = k.const_data_ptr();
  p.v = v.const_data_ptr();
  p.o = o.mutable_data_ptr();
  strides(q, p.q_stride_b, p.q_stride_h, p.q_stride_n);
  strides(k, p.k_stride_b, p.k_stride_h, p.k_stride_n);
  strides(v, p.v_stride_b, p.v_stride_h, p.v_stride_n);
  strides(o, p.o_stride_b, p.o_stride_h, p.o_stride_n);
  p.batch = (int32_t)q.size(0);
  p.heads_q = (int32_t)q.size(1);
  p.heads_kv = (int32_t)k.size(1);
  p.seqlen_q = (int32_t)q.size(2);
  p.seqlen_k = (int32_t)k.size(2);
  p.head_dim = (int32_t)q.size(3);
  p.scale = (float)(scale.has_value() ? *scale : 1.0 / std::sqrt((double)q.size(3)));
  p.causal = causal ? 1 : 0;
  p.dtype = p.kv_dtype = (decltype(p.dtype))dtype_code(q.scalar_type());
  void* stream = at::hip::getCurrentHIPStreamMasqueradingAsCUDA(q.device().index()).stream();
  auto workspace = [&](size_t bytes) { return at::empty({(int64_t)(bytes / 4)}, q.options().dtype(at::kFloat)); };

  const int64_t split_len = route(q.scalar_type() != at::kFloat, p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_k, p.head_dim);
  fa_status st;
  if (split_len > 0) {
    const size_t need = g_abi.splitk_workspace_bytes(p.batch, p.heads_q, p.seqlen_q, p.head_dim,
                                                     (int32_t)ceil_div(p.seqlen_k, split_len));
    const at::Tensor ws = workspace(need);
    st = g_abi.splitk(&p, (int32_t)split_len, ws.mutable_data_ptr(), need, stream);
  } else {
    const size_t need = g_abi.fwd_workspace_bytes(&p);
    const at::Tensor ws = need ? workspace(need) : at::Tensor();
    st = g_abi.fwd_ws(&p, need ? ws.mutable_data_ptr() : nullptr, need, stream);
  }
  TORCH_CHECK(st != FA_ERR_HIP, "fused_attn HIP ", split_len > 0 ? "attention_splitk" : "attention_fwd", " failed (HIP error): ",
              g_abi.last_error());
  // refused before anything was launched: the Python kernel reports it
  if (st != FA_OK) return call_python(c10::DispatchKey::CompositeExplicitAutograd, q, k, v, causal, scale);
  return o;
}

// Autograd: the op has no formula of its own, so a call that would record one goes to the Python kernel, which
// records the node that the op's users registered, or one that raises.
at::Tensor attention_autograd(c10::DispatchKeySet ks, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal,
                              std::optional<double> scale) {
  if (c10::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad()))
    return call_python(c10::DispatchKey::Autograd, q, k, v, causal, scale);
  using Fn = at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&, bool, std::optional<double>);
  static const auto op = attention_op().typed<Fn>();
  const at::AutoDispatchBelowAutograd below;
  return op.redispatch(ks & c10::after_autograd_keyset, q, k, v, causal, scale);
}

}  // namespace

extern "C" {

// What this library was built against: a torch build has no stable C++ ABI, and the HIP library bound below may come
// from elsewhere.  Python compares them before it registers the kernels, so loading the library has no effect.
const char* fa_torch_built_for(void) { return FA_TORCH_BUILD; }
int32_t fa_torch_abi_version(void) { return FA_ABI_VERSION; }
size_t fa_torch_params_size(void) { return sizeof(fa_fwd_params); }

// Registers the kernels, once; 0 when torch refuses them.
int32_t fa_torch_register(void) {
  try {
    static torch::Library cuda(torch::Library::IMPL, "fused_attn", c10::DispatchKey::CUDA, __FILE__, __LINE__);
    static torch::Library autograd(torch::Library::IMPL, "fused_attn", c10::DispatchKey::AutogradCUDA, __FILE__, __LINE__);
    static const bool once = (cuda.impl("attention", TORCH_FN(attention_gpu)), autograd.impl("attention", TORCH_FN(attention_autograd)), true);
    return once;
  } catch (const std::exception&) {
    return 0;
  }
}

void fa_torch_bind(void* fwd_workspace_bytes, void* fwd_ws, void* splitk_workspace_bytes, void* splitk, void* last_error) {
  g_abi.fwd_workspace_bytes = (decltype(g_abi.fwd_workspace_bytes))fwd_workspace_bytes;
  g_abi.fwd_ws = (decltype(g_abi.fwd_ws))fwd_ws;
  g_abi.splitk_workspace_bytes = (decltype(g_abi.splitk_workspace_bytes))splitk_workspace_bytes;
  g_abi.splitk = (decltype(g_abi.splitk))splitk;
  g_abi.last_error = (decltype(g_abi.last_error))last_error;
}

// Device `index` runs the library bound above (which happens before).
void fa_torch_enable(int32_t index) {
  if (index >= 0 && index < 64) g_devices.fetch_or(uint64_t{1} << index, std::memory_order_release);
}

int32_t fa_torch_backend_forced(void) { return backend_forced(); }

int64_t fa_torch_route(int32_t half, int64_t b, int64_t hq, int64_t hkv, int64_t nq, int64_t nk, int64_t d) {
  return route(half != 0, b, hq, hkv, nq, nk, d);
}

}  // extern "C"
