"""PyTorch custom ops (namespace `nvhip`) over the C-ABI kernels of libnvhip.so.

Each op has a CUDA (= ROCm/HIP device) implementation that allocates its outputs with torch's caching allocator and
launches the kernel on torch's current stream (csrc/torch_ops.cpp, libnvhip_torch.so), and a fake (meta) implementation
here so torch.compile and graph capture can trace it. There is no CPU implementation: CPU tensors raise in the
dispatcher.

The user-facing functions with the reference's signatures are in nanovllm_hip.kernels; these ops take the already
validated, normalised arguments.
"""
import os

import torch

from nanovllm_hip import _lib

_DEF = torch.library.Library("nvhip", "DEF")

_DEF.define(
    "qk_norm_rope_kv(Tensor q, Tensor k, Tensor v, Tensor positions, Tensor q_weight, Tensor k_weight, float eps, "
    "Tensor cos_sin_cache, Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor? slot_mapping, bool write_k) "
    "-> (Tensor, Tensor)")
_DEF.define("rms_norm(Tensor x, Tensor w, float eps) -> Tensor")
_DEF.define("fused_add_rms_norm(Tensor x, Tensor residual, Tensor w, float eps) -> (Tensor, Tensor)")
_DEF.define("fused_add_rms_norm_(Tensor x, Tensor(a!) residual, Tensor w, float eps) -> Tensor")
_DEF.define("silu_and_mul(Tensor x) -> Tensor")
_DEF.define("matmul(Tensor a, Tensor b, str input_precision) -> Tensor")
_DEF.define("matmul_silu_mul(Tensor a, Tensor w) -> Tensor")
_DEF.define("rms_norm_matmul(Tensor x, Tensor? residual, Tensor norm_w, float eps, Tensor w, bool silu) "
            "-> (Tensor, Tensor)")
_DEF.define("matmul_add_rms_norm(Tensor x, Tensor w, Tensor residual, Tensor norm_w, float eps) -> (Tensor, Tensor)")
_DEF.define("qk_norm_rope_kv_decode_attention(Tensor q, Tensor k, Tensor v, Tensor positions, Tensor q_w, Tensor k_w, "
            "float eps, Tensor cos_sin, Tensor(a!) k_cache, Tensor(b!) v_cache, Tensor slot_mapping, "
            "Tensor cache_seqlens, Tensor block_table, float scale) -> Tensor")
_DEF.define("prefill_attention(Tensor q, Tensor k, Tensor v, Tensor cu_seqlens_q, Tensor cu_seqlens_k, "
            "int max_seqlen_q, int max_seqlen_k, float scale, bool causal, Tensor? block_table) -> Tensor")
_DEF.define("prefill_attention_out(Tensor q, Tensor k, Tensor v, Tensor cu_seqlens_q, Tensor cu_seqlens_k, "
            "int max_seqlen_q, int max_seqlen_k, float scale, bool causal, Tensor? block_table, "
            "Tensor(a!) out) -> ()")
_DEF.define("store_kvcache(Tensor key, Tensor value, Tensor(a!) k_cache, Tensor(b!) v_cache, "
            "Tensor slot_mapping) -> ()")
_DEF.define("paged_decode_attention(Tensor q, Tensor k_cache, Tensor v_cache, Tensor block_table, "
            "Tensor context_lens, int q_len, float scale, bool causal) -> Tensor")
_DEF.define("argmax(Tensor logits) -> Tensor")

_OPS = ("qk_norm_rope_kv", "rms_norm", "fused_add_rms_norm", "fused_add_rms_norm_", "silu_and_mul", "matmul",
        "matmul_silu_mul", "rms_norm_matmul", "matmul_add_rms_norm", "qk_norm_rope_kv_decode_attention",
        "prefill_attention", "prefill_attention_out", "store_kvcache", "paged_decode_attention", "argmax")


def _load():
    """Loads the native implementations; without the built libraries every op raises when it is called."""
    if os.path.exists(_lib.LIB_PATH) and os.path.exists(_lib.TORCH_LIB_PATH):
        _lib.lib()  # libnvhip.so first: its path and ABI version are checked here
        torch.ops.load_library(_lib.TORCH_LIB_PATH)
        return

    def missing(*args):
        raise RuntimeError(f"{_lib.LIB_PATH} and {_lib.TORCH_LIB_PATH} are not both built: run `make -C <package>/csrc` "
                           f"(or __graft_entry__.build())")
    for name in _OPS:
        _DEF.impl(name, missing, "CUDA")


_load()


# ------------------------------------------------------------------ qk_norm_rope_kv

def _qk_outputs(q, k, write_k):
    T, Hq, D = q.shape
    q_out = q.new_empty((T, Hq, D))
    k_out = k.new_empty((T, k.shape[1], D)) if write_k else k.new_empty((0,))
    return q_out, k_out


@torch.library.register_fake("nvhip::qk_norm_rope_kv")
def _qk_norm_rope_kv_fake(q, k, v, positions, q_weight, k_weight, eps, cos_sin_cache, k_cache, v_cache,
                          slot_mapping, write_k):
    return _qk_outputs(q, k, write_k)


# ------------------------------------------------------------------ rms_norm / fused_add_rms_norm

@torch.library.register_fake("nvhip::rms_norm")
def _rms_norm_fake(x, w, eps):
    return torch.empty(x.shape, dtype=x.dtype, device=x.device)


@torch.library.register_fake("nvhip::fused_add_rms_norm")
def _fused_add_rms_norm_fake(x, residual, w, eps):
    return torch.empty(x.shape, dtype=x.dtype, device=x.device), torch.empty(x.shape, dtype=x.dtype, device=x.device)


@torch.library.register_fake("nvhip::fused_add_rms_norm_")
def _fused_add_rms_norm_inplace_fake(x, residual, w, eps):
    return torch.empty(x.shape, dtype=x.dtype, device=x.device)


# ------------------------------------------------------------------ silu_and_mul

@torch.library.register_fake("nvhip::silu_and_mul")
def _silu_and_mul_fake(x):
    return torch.empty((x.shape[0], x.shape[1] // 2), dtype=x.dtype, device=x.device)


# ------------------------------------------------------------------ matmul

@torch.library.register_fake("nvhip::matmul")
def _matmul_fake(a, b, input_precision):
    return torch.empty((a.shape[0], b.shape[1]), dtype=a.dtype, device=a.device)


# ------------------------------------------------------------------ paged decode attention

@torch.library.register_fake("nvhip::paged_decode_attention")
def _paged_decode_attention_fake(q, k_cache, v_cache, block_table, context_lens, q_len, scale, causal):
    return torch.empty(q.shape, dtype=q.dtype, device=q.device)


# ------------------------------------------------------------------ store_kvcache

@torch.library.register_fake("nvhip::store_kvcache")
def _store_kvcache_fake(key, value, k_cache, v_cache, slot_mapping):
    return None


# ------------------------------------------------------------------ GEMM + SiLU x Mul epilogue

@torch.library.register_fake("nvhip::matmul_silu_mul")
def _matmul_silu_mul_fake(a, w):
    return torch.empty((a.shape[0], w.shape[0] // 2), dtype=a.dtype, device=a.device)


# ------------------------------------------------------------------ RMSNorm / Add+RMSNorm fused into the next GEMM

@torch.library.register_fake("nvhip::rms_norm_matmul")
def _rms_norm_matmul_fake(x, residual, norm_w, eps, w, silu):
    N = w.shape[0] // 2 if silu else w.shape[0]
    out = torch.empty((x.shape[0], N), dtype=x.dtype, device=x.device)
    return out, (torch.empty_like(x) if residual is not None else x.new_empty((0,)))


# ------------------------------------------------------------------ GEMM followed by the Add+RMSNorm that consumes it

@torch.library.register_fake("nvhip::matmul_add_rms_norm")
def _matmul_add_rms_norm_fake(x, w, residual, norm_w, eps):
    out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
    return out, torch.empty_like(out)


# ------------------------------------------------------------------ fused q/k norm + RoPE + KV write + decode attention

@torch.library.register_fake("nvhip::qk_norm_rope_kv_decode_attention")
def _qk_norm_rope_kv_decode_attention_fake(q, k, v, positions, q_w, k_w, eps, cos_sin, k_cache, v_cache,
                                           slot_mapping, cache_seqlens, block_table, scale):
    return torch.empty(q.shape, dtype=q.dtype, device=q.device)


# ------------------------------------------------------------------ prefill (varlen) attention

@torch.library.register_fake("nvhip::prefill_attention")
def _prefill_attention_fake(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, scale, causal,
                            block_table):
    return torch.empty(q.shape, dtype=q.dtype, device=q.device)


# ------------------------------------------------------------------ greedy sampling (argmax over the vocabulary)

@torch.library.register_fake("nvhip::argmax")
def _argmax_fake(logits):
    return torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
