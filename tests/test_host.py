"""Host-side behaviour of the Python layer (CPU only): the reference's argument assertions, output shapes through
the ops' fake (meta) implementations, and no CPU fallback (CPU tensors are refused by the dispatcher)."""
import pathlib
import re

import numpy as np
import pytest
import torch

from nanovllm_hip.kernels import fused_add_rms_norm, matmul, qk_norm_rope_kv, rms_norm, silu_and_mul

BF16 = torch.bfloat16


def qk_args(device="meta", T=5, Hq=16, Hkv=8, D=128, store=True, dtype=BF16):
    qkv = torch.empty(T, (Hq + 2 * Hkv) * D + 64, dtype=dtype, device=device)
    q = qkv[:, :Hq * D].view(T, Hq, D)
    k = qkv[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D)
    v = qkv[:, (Hq + Hkv) * D:(Hq + 2 * Hkv) * D].view(T, Hkv, D)
    cache = (torch.empty(4, 256, Hkv, D, dtype=BF16, device=device) if store
             else torch.empty(0, device=device))
    return dict(q=q, k=k, v=v, positions=torch.empty(T, dtype=torch.int64, device=device),
                q_weight=torch.empty(D, dtype=BF16, device=device), k_weight=torch.empty(D, dtype=BF16, device=device),
                eps=1e-6, cos_sin_cache=torch.empty(40960, 1, D, device=device), k_cache=cache,
                v_cache=cache.clone() if store else cache,
                slot_mapping=torch.empty(T, dtype=torch.int32, device=device) if store else None, write_k=True)


def test_qk_shapes_through_fake_impl():
    q_out, k_out = qk_norm_rope_kv(**qk_args())
    assert q_out.shape == (5, 16, 128) and k_out.shape == (5, 8, 128) and q_out.is_contiguous()
    a = qk_args()
    a["write_k"] = False
    assert qk_norm_rope_kv(**a)[1] is None
    q_out, k_out = qk_norm_rope_kv(**qk_args(store=False))
    assert q_out.shape == (5, 16, 128)


@pytest.mark.parametrize("bad", ["dtype", "head_dim", "gqa", "stride", "positions", "cache", "slots", "table"])
def test_qk_assertions(bad):
    a = qk_args()
    if bad == "dtype":
        a = qk_args(dtype=torch.float16)
    elif bad == "head_dim":
        a = qk_args(D=96)
    elif bad == "gqa":
        a = qk_args(Hq=12, Hkv=8)
    elif bad == "stride":
        a["q"] = torch.empty(5, 128, 16, dtype=BF16, device="meta").transpose(1, 2)
    elif bad == "positions":
        a["positions"] = a["positions"].to(torch.int32)
    elif bad == "cache":
        a["k_cache"] = torch.empty(4, 256, 8, 256, dtype=BF16, device="meta")[..., :128]
    elif bad == "slots":
        a["slot_mapping"] = None
    elif bad == "table":
        a["cos_sin_cache"] = torch.empty(40960, 1, 128, dtype=BF16, device="meta")
    with pytest.raises(AssertionError):
        qk_norm_rope_kv(**a)


def test_norm_silu_matmul_shapes_and_assertions():
    x = torch.empty(7, 1024, dtype=BF16, device="meta")
    w = torch.empty(1024, dtype=BF16, device="meta")
    assert rms_norm(x, w, 1e-6).shape == (7, 1024)
    assert rms_norm(torch.empty(7, 16, 128, dtype=BF16, device="meta"), w[:128], 1e-6).shape == (7, 16, 128)
    y, s = fused_add_rms_norm(x, x, w, 1e-6)
    assert y.shape == s.shape == (7, 1024)
    assert silu_and_mul(torch.empty(7, 6144, dtype=BF16, device="meta")).shape == (7, 3072)
    a = torch.empty(32, 1024, dtype=BF16, device="meta")
    b = torch.empty(4096, 1024, dtype=BF16, device="meta").t()
    assert matmul(a, b).shape == (32, 4096)
    with pytest.raises(AssertionError):
        fused_add_rms_norm(x, torch.empty(7, 512, dtype=BF16, device="meta"), w, 1e-6)
    with pytest.raises(AssertionError):
        rms_norm(x.float(), w, 1e-6)
    with pytest.raises(AssertionError):
        matmul(a, b.float())
    with pytest.raises(AssertionError):
        matmul(a, b, input_precision="bf16x3")
    with pytest.raises(AssertionError):
        matmul(a, torch.empty(512, 4096, dtype=BF16, device="meta"))


def test_no_cpu_fallback():
    """The ops have no CPU kernel: CPU tensors fail loudly in the dispatcher instead of running a slow path."""
    x = torch.randn(4, 256).to(BF16)
    w = torch.ones(256, dtype=BF16)
    with pytest.raises(NotImplementedError):
        rms_norm(x, w, 1e-6)
    with pytest.raises(NotImplementedError):
        silu_and_mul(x)
    with pytest.raises(NotImplementedError):
        matmul(x, x.t())
    with pytest.raises(NotImplementedError):
        qk_norm_rope_kv(**qk_args(device="cpu"))


def test_model_latches_the_kernel_backend_at_construction():
    # the reference's layers read nanovllm.kernels.backend once, in __init__ (layers/layernorm.py:18); so does the
    # harness model, and a later change of the module value does not reach a model already built
    import nanovllm_hip.kernels as kernels
    from nanovllm_hip.harness.qwen3 import Qwen3, Qwen3Config
    cfg = Qwen3Config(vocab_size=64, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1, head_dim=64, max_position_embeddings=16)
    old = kernels.backend
    try:
        kernels.backend = "compile"
        model = Qwen3(cfg, "meta")
        kernels.backend = "hip"
        assert model.kernel_backend == "torch"
        assert Qwen3(cfg, "meta").kernel_backend == "hip"
        assert Qwen3(cfg, "meta", kernel_backend="compile").kernel_backend == "torch"
        kernels.backend = "triton"
        with pytest.raises(ValueError):
            Qwen3(cfg, "meta")
    finally:
        kernels.backend = old


def test_every_op_has_its_native_implementation():
    from nanovllm_hip import ops
    defined = {s.name for s in torch._C._jit_get_all_schemas() if s.name.startswith("nvhip::")}
    assert defined == {f"nvhip::{name}" for name in ops._OPS}
    for name in ops._OPS:
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"nvhip::{name}", "CUDA"), name


def test_no_asm_writes_m0_itself():
    """The compiler keeps values of its own in m0 and cannot be told that an asm statement overwrites it (it is a
    reserved register in a clobber list): a statement that needs a value there takes it as an operand in m0."""
    csrc = pathlib.Path(__file__).resolve().parent.parent / "nano-vllm-triton-kernels_amd" / "csrc"
    operands = 0
    for path in sorted(csrc.glob("*.hip")) + sorted(csrc.glob("*.h")):
        for statement in re.findall(r"asm\s+volatile\s*\((.*?)\);", path.read_text(), re.S):
            assert not re.search(r"\bm0\s*,", statement), (path.name, statement)
            operands += '"{m0}"' in statement
    assert operands == 2  # the loads into LDS of gemm_stream_nt and prefill_wide_kernel


def test_fast_silu_window_holds_its_error():
    """silu_bf16_n takes the exact form where its fast one is near a bf16 tie: the window has to hold the largest
    distance of the two over all bf16 gates below 8, the hardware exp and reciprocal and expf each off by up to an ulp."""
    common = pathlib.Path(__file__).resolve().parent.parent / "nano-vllm-triton-kernels_amd" / "csrc" / "common.h"
    low, width = (int(x, 0) for x in re.search(r"& 0xffffu\) - (\w+)u <= (\w+)u", common.read_text()).groups())
    window = min(0x8000 - low, low + width - 0x8000)
    f32 = np.float32
    g = (np.arange(65536, dtype=np.uint32) << 16).view(f32)
    g = g[np.abs(g) < 8]
    bits = lambda x: x.astype(f32).view(np.int32).astype(np.int64)
    off = lambda x, ulps: (bits(x) + ulps).astype(np.int32).view(f32)
    t = (g * f32(-1.44269504)).astype(f32)
    exact = [bits(g / (f32(1) + off(np.exp(-g.astype(np.float64)), a))) for a in (-1, 0, 1)]
    worst = 0
    for a in (-1, 0, 1):
        rcp = 1 / (f32(1) + off(np.exp2(t.astype(np.float64)), a)).astype(np.float64)
        for b in (-1, 0, 1):
            fast = bits(g * off(rcp, b))
            worst = max(worst, *(int(np.abs(fast - x).max()) for x in exact))
    assert 6 < worst <= window, (worst, window)
