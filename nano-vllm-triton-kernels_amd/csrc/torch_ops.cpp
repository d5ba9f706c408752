// The CUDA (= ROCm/HIP device) implementations of the `nvhip` torch custom ops (their schemas and fake implementations
// are in nanovllm_hip/ops.py): output allocation with torch's caching allocator and the launch of the C-ABI kernel of
// libnvhip.so on torch's current stream of the tensors' device. The arguments were validated by nanovllm_hip.kernels.
//
// Native because a call is mostly host time: a Python implementation that passes ~20 arguments through ctypes took
// 12-15 us per call, more than the kernels of a decode step of one request.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <algorithm>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "nvhip.h"

namespace {

using at::Tensor;

// Raises what nanovllm_hip._lib.check raises: ValueError (bad argument) or KernelError (launch failure).
void check(int status, const char* what) {
  if (status == NVHIP_OK) return;
  const char* text = nvhip_last_error();
  const std::string msg = text && *text ? text : what;
  TORCH_CHECK_VALUE(status != NVHIP_EINVAL, msg);
  pybind11::gil_scoped_acquire gil;
  const pybind11::object error = pybind11::module_::import("nanovllm_hip._lib").attr("KernelError");
  PyErr_SetString(error.ptr(), msg.c_str());
  python_error e;
  e.persist();
  throw e;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int32_t* i32(const Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); }
int64_t* i64(const Tensor& t) { return static_cast<int64_t*>(t.data_ptr()); }

// The attention workspaces (decode and prefill): they start with the decode attention's per-pair counters, which must
// be zero before a call and which every call leaves zero, so one workspace is zero-filled once and kept per device,
// for both ops (a graph captured after an eager warm-up call reuses it, so the zero fill is not captured). Attention
// calls on one device must therefore not run concurrently on unordered streams. A workspace is never freed: a
// captured graph keeps using its address (a larger need adds a new one).
void* attention_workspace(const Tensor& q, int64_t nbytes) {
  if (nbytes <= 0) return nullptr;
  static std::mutex lock;
  static auto* const all = new std::unordered_map<int, std::vector<Tensor>>();
  const std::lock_guard<std::mutex> guard(lock);
  std::vector<Tensor>& held = (*all)[q.device().index()];
  if (held.empty() || held.back().numel() < nbytes) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const hipError_t rc = hipStreamIsCapturing(static_cast<hipStream_t>(stream_of(q)), &capture);
    // a zero fill recorded into the graph would run only at replay, after eager calls that already used the new
    // workspace's uninitialised counters
    TORCH_CHECK(rc == hipSuccess && capture == hipStreamCaptureStatusNone, "nvhip attention: a ", nbytes,
                "-byte workspace is needed inside a graph capture, but the workspace held for this device is ",
                held.empty() ? 0 : held.back().numel(), " bytes; run the same call once eagerly before capturing it");
    held.push_back(at::zeros({std::max<int64_t>(nbytes, int64_t(1) << 20)}, q.options().dtype(at::kByte)));
  }
  return held.back().data_ptr();
}

std::tuple<Tensor, Tensor> qk_norm_rope_kv(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& positions,
                                           const Tensor& q_weight, const Tensor& k_weight, double eps,
                                           const Tensor& cos_sin, const Tensor& k_cache, const Tensor& v_cache,
                                           const std::optional<Tensor>& slot_mapping, bool write_k) {
  const c10::DeviceGuard guard(q.device());
  const int64_t T = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
  Tensor q_out = at::empty({T, Hq, D}, q.options());
  Tensor k_out = write_k ? at::empty({T, Hkv, D}, k.options()) : at::empty({0}, k.options());
  const bool store = k_cache.numel() > 0;
  check(nvhip_qk_norm_rope_kv_bf16(q_out.data_ptr(), write_k ? k_out.data_ptr() : nullptr, q.data_ptr(), k.data_ptr(),
                                   v.data_ptr(), q.stride(0), k.stride(0), v.stride(0), i64(positions),
                                   store ? i32(*slot_mapping) : nullptr, q_weight.data_ptr(), k_weight.data_ptr(),
                                   static_cast<float*>(cos_sin.data_ptr()), cos_sin.stride(0), cos_sin.size(0),
                                   store ? k_cache.data_ptr() : nullptr, store ? v_cache.data_ptr() : nullptr,
                                   store ? k_cache.numel() / (Hkv * D) : 0, T, Hq, Hkv, D, float(eps), stream_of(q)),
        "qk_norm_rope_kv");
  return {q_out, k_out};
}

Tensor rms_norm(const Tensor& x, const Tensor& w, double eps) {
  const c10::DeviceGuard guard(x.device());
  const bool flat = x.dim() == 2;
  Tensor y = at::empty(x.sizes(), x.options());
  check(nvhip_rms_norm_bf16(y.data_ptr(), x.data_ptr(), w.data_ptr(), x.size(0), flat ? 1 : x.size(1), x.stride(0),
                            flat ? 0 : x.stride(1), x.size(-1), float(eps), stream_of(x)),
        "rms_norm");
  return y;
}

Tensor add_rms(const Tensor& x, const Tensor& residual, const Tensor& w, double eps, const Tensor& res_out) {
  Tensor y = at::empty(x.sizes(), x.options());
  check(nvhip_add_rms_norm_bf16(y.data_ptr(), res_out.data_ptr(), x.data_ptr(), residual.data_ptr(), w.data_ptr(),
                                x.size(0), x.stride(0), residual.stride(0), x.size(1), float(eps), stream_of(x)),
        "fused_add_rms_norm");
  return y;
}

std::tuple<Tensor, Tensor> fused_add_rms_norm(const Tensor& x, const Tensor& residual, const Tensor& w, double eps) {
  const c10::DeviceGuard guard(x.device());
  Tensor s = at::empty(x.sizes(), x.options());
  return {add_rms(x, residual, w, eps, s), s};
}

Tensor fused_add_rms_norm_(const Tensor& x, const Tensor& residual, const Tensor& w, double eps) {
  const c10::DeviceGuard guard(x.device());
  return add_rms(x, residual, w, eps, residual);
}

Tensor silu_and_mul(const Tensor& x) {
  const c10::DeviceGuard guard(x.device());
  const int64_t rows = x.size(0), n = x.size(1) / 2;
  Tensor out = at::empty({rows, n}, x.options());
  check(nvhip_silu_mul_bf16(out.data_ptr(), x.data_ptr(), rows, x.stride(0), n, stream_of(x)), "silu_and_mul");
  return out;
}

Tensor matmul(const Tensor& a, const Tensor& b, c10::string_view input_precision) {
  const c10::DeviceGuard guard(a.device());
  const int64_t M = a.size(0), K = a.size(1), N = b.size(1);
  Tensor c = at::empty({M, N}, a.options());
  check(nvhip_matmul(c.data_ptr(), a.data_ptr(), b.data_ptr(), M, N, K, a.stride(0), a.stride(1), b.stride(0),
                     b.stride(1), c.stride(0), c.stride(1),
                     a.scalar_type() == at::kBFloat16 ? NVHIP_DTYPE_BF16 : NVHIP_DTYPE_F32,
                     input_precision == "tf32" ? NVHIP_PREC_TF32 : NVHIP_PREC_IEEE, stream_of(a)),
        "matmul");
  return c;
}

Tensor matmul_silu_mul(const Tensor& a, const Tensor& w) {
  const c10::DeviceGuard guard(a.device());
  const int64_t M = a.size(0), K = a.size(1), n = w.size(0) / 2;
  Tensor out = at::empty({M, n}, a.options());
  check(nvhip_matmul_silu_mul_bf16(out.data_ptr(), a.data_ptr(), w.data_ptr(), M, n, K, a.stride(0), w.stride(0),
                                   out.stride(0), stream_of(a)),
        "matmul_silu_mul");
  return out;
}

std::tuple<Tensor, Tensor> rms_norm_matmul(const Tensor& x, const std::optional<Tensor>& residual,
                                           const Tensor& norm_w, double eps, const Tensor& w, bool silu) {
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = silu ? w.size(0) / 2 : w.size(0);
  const bool add = residual.has_value();
  Tensor out = at::empty({M, N}, x.options());
  Tensor res_out = add ? at::empty({M, K}, x.options()) : at::empty({0}, x.options());
  check(nvhip_rms_norm_matmul_bf16(out.data_ptr(), add ? res_out.data_ptr() : nullptr, x.data_ptr(),
                                   add ? residual->data_ptr() : nullptr, norm_w.data_ptr(), float(eps), w.data_ptr(), M,
                                   N, K, x.stride(0), add ? residual->stride(0) : 0, w.stride(0), out.stride(0),
                                   int(silu), stream_of(x)),
        "rms_norm_matmul");
  return {out, res_out};
}

std::tuple<Tensor, Tensor> matmul_add_rms_norm(const Tensor& x, const Tensor& w, const Tensor& residual,
                                               const Tensor& norm_w, double eps) {
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  Tensor y = at::empty({M, N}, x.options()), res_out = at::empty({M, N}, x.options());
  const int64_t need = nvhip_matmul_add_rms_norm_workspace_size(M, N, K);
  Tensor ws = at::empty({(std::max<int64_t>(need, 16) + 3) / 4}, x.options().dtype(at::kFloat));
  check(nvhip_matmul_add_rms_norm_bf16(y.data_ptr(), res_out.data_ptr(), x.data_ptr(), w.data_ptr(),
                                       residual.data_ptr(), norm_w.data_ptr(), float(eps), M, N, K, x.stride(0),
                                       w.stride(0), ws.data_ptr(), ws.numel() * 4, stream_of(x)),
        "matmul_add_rms_norm");
  return {y, res_out};
}

Tensor qk_norm_rope_kv_decode_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& positions,
                                        const Tensor& q_w, const Tensor& k_w, double eps, const Tensor& cos_sin,
                                        const Tensor& k_cache, const Tensor& v_cache, const Tensor& slot_mapping,
                                        const Tensor& cache_seqlens, const Tensor& block_table, double scale) {
  const c10::DeviceGuard guard(q.device());
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2), num_blocks = k_cache.size(0), bs = k_cache.size(1),
                Hkv = k_cache.size(2), max_blocks = block_table.size(1);
  Tensor out = at::empty({B, Hq, D}, q.options());
  const int64_t need = nvhip_paged_decode_attention_workspace_size(B, 1, Hq, Hkv, D, bs, max_blocks);
  void* ws = attention_workspace(q, need);
  check(nvhip_qk_norm_rope_kv_decode_attention_bf16(
            out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), k.stride(0), v.stride(0),
            i64(positions), i32(slot_mapping), q_w.data_ptr(), k_w.data_ptr(),
            static_cast<float*>(cos_sin.data_ptr()), cos_sin.stride(0), cos_sin.size(0), float(eps),
            k_cache.data_ptr(), v_cache.data_ptr(), i32(block_table), i32(cache_seqlens), B, Hq, Hkv, D, bs,
            num_blocks, max_blocks, out.stride(0), out.stride(1), float(scale), ws, ws ? need : 0, stream_of(q)),
        "qk_norm_rope_kv_decode_attention");
  return out;
}

// Writes the attention into out [Tq, Hq, D] (rows of Hq * D contiguous heads: out.stride(2) == 1).
void prefill_attention_out(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k,
                           int64_t max_q, int64_t max_k, double scale, bool causal,
                           const std::optional<Tensor>& block_table, const Tensor& out) {
  const c10::DeviceGuard guard(q.device());
  const int64_t Tq = q.size(0), Hq = q.size(1), D = q.size(2), num_seqs = cu_q.size(0) - 1;
  const bool paged = block_table.has_value();
  const int64_t Hkv = paged ? k.size(2) : k.size(1);
  const int64_t need = nvhip_prefill_attention_workspace_size(num_seqs, max_q, max_k, Hq, Hkv, D, Tq);
  void* ws = attention_workspace(q, need);
  check(nvhip_prefill_attention_bf16(
            out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), i32(cu_q), i32(cu_k), num_seqs, max_q, max_k, Tq,
            Hq, Hkv, D, q.stride(0), q.stride(1), paged ? Hkv * D : k.stride(0), paged ? Hkv * D : v.stride(0),
            out.stride(0), out.stride(1), paged ? i32(*block_table) : nullptr, paged ? k.size(1) : 0,
            paged ? k.size(0) : 0, paged ? block_table->size(1) : 0, float(scale), int(causal), ws, ws ? need : 0,
            stream_of(q)),
        "prefill_attention");
}

Tensor prefill_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k,
                         int64_t max_q, int64_t max_k, double scale, bool causal,
                         const std::optional<Tensor>& block_table) {
  Tensor out = at::empty(q.sizes(), q.options());
  prefill_attention_out(q, k, v, cu_q, cu_k, max_q, max_k, scale, causal, block_table, out);
  return out;
}

void store_kvcache(const Tensor& key, const Tensor& value, const Tensor& k_cache, const Tensor& v_cache,
                   const Tensor& slot_mapping) {
  const c10::DeviceGuard guard(key.device());
  const int64_t n = key.size(0), row = key.size(1) * key.size(2);
  check(nvhip_store_kvcache(k_cache.data_ptr(), v_cache.data_ptr(), key.data_ptr(), value.data_ptr(), key.stride(0),
                            value.stride(0), i32(slot_mapping), row ? k_cache.numel() / row : 0, n, row,
                            key.element_size(), stream_of(key)),
        "store_kvcache");
}

Tensor paged_decode_attention(const Tensor& q, const Tensor& k_cache, const Tensor& v_cache, const Tensor& block_table,
                              const Tensor& context_lens, int64_t q_len, double scale, bool causal) {
  const c10::DeviceGuard guard(q.device());
  const int64_t T = q.size(0), Hq = q.size(1), D = q.size(2), num_blocks = k_cache.size(0), bs = k_cache.size(1),
                Hkv = k_cache.size(2), num_seqs = context_lens.size(0), max_blocks = block_table.size(1);
  Tensor out = at::empty({T, Hq, D}, q.options());
  const int64_t need = nvhip_paged_decode_attention_workspace_size(num_seqs, q_len, Hq, Hkv, D, bs, max_blocks);
  void* ws = attention_workspace(q, need);
  check(nvhip_paged_decode_attention_bf16(out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                                          i32(block_table), i32(context_lens), num_seqs, q_len, Hq, Hkv, D, bs,
                                          num_blocks, max_blocks, q.stride(0), q.stride(1), out.stride(0),
                                          out.stride(1), float(scale), int(causal), ws, ws ? need : 0, stream_of(q)),
        "paged_decode_attention");
  return out;
}

Tensor argmax(const Tensor& logits) {
  const c10::DeviceGuard guard(logits.device());
  const int64_t rows = logits.size(0), n = logits.size(1);
  Tensor out = at::empty({rows}, logits.options().dtype(at::kLong));
  const int64_t need = nvhip_argmax_workspace_size(rows, n);
  Tensor ws = at::empty({std::max<int64_t>(need, 16)}, logits.options().dtype(at::kByte));
  check(nvhip_argmax_bf16(i64(out), logits.data_ptr(), rows, n, logits.stride(0), ws.data_ptr(), need,
                          stream_of(logits)),
        "argmax");
  return out;
}

}  // namespace

TORCH_LIBRARY_IMPL(nvhip, CUDA, m) {
  m.impl("qk_norm_rope_kv", qk_norm_rope_kv);
  m.impl("rms_norm", rms_norm);
  m.impl("fused_add_rms_norm", fused_add_rms_norm);
  m.impl("fused_add_rms_norm_", fused_add_rms_norm_);
  m.impl("silu_and_mul", silu_and_mul);
  m.impl("matmul", matmul);
  m.impl("matmul_silu_mul", matmul_silu_mul);
  m.impl("rms_norm_matmul", rms_norm_matmul);
  m.impl("matmul_add_rms_norm", matmul_add_rms_norm);
  m.impl("qk_norm_rope_kv_decode_attention", qk_norm_rope_kv_decode_attention);
  m.impl("prefill_attention", prefill_attention);
  m.impl("prefill_attention_out", prefill_attention_out);
  m.impl("store_kvcache", store_kvcache);
  m.impl("paged_decode_attention", paged_decode_attention);
  m.impl("argmax", argmax);
}
