"""ctypes bindings for ``libvdamd_ops.so`` (the gfx950 kernel library).

Every entry point takes raw device pointers plus the current HIP stream, so
the launches are captured when the caller is inside a hipGraph capture.
Shapes are validated here, on the host, before a kernel is launched: an
out-of-bounds access in a hand-written kernel can take the GPU down.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
from ctypes import c_float, c_int, c_long, c_void_p
from typing import Optional, Tuple

import torch

from ..logger import init_logger

logger = init_logger(__name__)
_LIB: Optional[ctypes.CDLL] = None
# VDAMD_OPS_LIB selects another build of the library (the host-sanitizer preset of build.py)
_LIB_PATH = os.environ.get("VDAMD_OPS_LIB") or os.path.join(
    os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "_C", "libvdamd_ops.so")
_DT = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}
MAX_SPLITS = 16


def load() -> ctypes.CDLL:
    global _LIB, MAX_SPLITS
    if _LIB is not None:
        return _LIB
    if not os.path.exists(_LIB_PATH):
        raise FileNotFoundError(f"{_LIB_PATH} is missing: run `python -m vllm_distributed_amd.build`")
    lib = ctypes.CDLL(_LIB_PATH)
    P, I, L, F = c_void_p, c_int, c_long, c_float
    sigs = {
        "vdamd_rms_norm": [P, P, P, P, F, I, I, L, L, I, P],
        "vdamd_layer_norm": [P, P, P, P, F, I, I, I, P],
        "vdamd_reduce_add_rms_norm": [P, P, I, P, P, F, I, I, L, I, P],
        "vdamd_silu_and_mul": [P, P, L, I, I, P],
        "vdamd_embedding": [P, P, P, I, I, I, I, I, P],
        "vdamd_mid_gemm": [P, L, P, L, P, L, P, P, I, I, I, I, I, I, I, I, P],
        "vdamd_mid_gemm_grouped": [P, L, P, L, P, L, L, P, I, P, I, I, I, I, I, I, I, I, P],
        "vdamd_stream_gemm": [P, L, P, L, P, L, P, P, L, I, I, I, I, I, I, I, I, I, P],
        "vdamd_big_gemm": [P, L, P, L, P, L, P, L, I, I, I, I, I, I, P],
        "vdamd_big_gemm_grouped": [P, L, P, L, P, L, L, P, I, P, I, I, I, I, I, I, P],
        "vdamd_rope_cache": [P, P, P, P, L, L, L, P, P, P, P, I, I, I, I, I, I, P, P, F, I, I, P, P, P],
        "vdamd_rope_cache_slabs": [P, P, I, P, L, P, P, P, P, I, I, I, I, I, P, P, F, I, I, P, P, P],
        "vdamd_paged_attention_decode": [P, P, P, L, P, P, P, I, P, F, I, I, I, I, I, I, L, I, I, P, P, I, F, P, P, L, P],
        "vdamd_paged_attention_prefill": [P, P, L, P, P, P, I, P, P, F, I, I, I, I, I, I, L, I, I, P, P, I, F, P, P, P],
        "vdamd_argmax": [P, P, I, I, L, I, P],
        "vdamd_sample": [P, P, I, I, L, P, P, P, P, P, I, P],
        "vdamd_w4a16_gemm": [P, L, P, L, P, P, P, I, I, I, I, I, I, I, P],
        "vdamd_w4_dequant": [P, P, P, I, I, I, I, P],
        "vdamd_skinny_gemm": [P, L, P, L, P, L, P, I, I, I, I, I, I, L, P],
        "vdamd_dynamic_fp8_quant": [P, P, P, I, I, L, I, P],
        "vdamd_w4a16_gemm_grouped": [P, L, P, L, P, P, L, L, P, I, I, I, I, I, I, I, P],
        "vdamd_moe_topk": [P, L, P, P, I, I, I, I, I, P],
        "vdamd_moe_align": [P, I, I, I, I, I, I, P, P, P, I, P],
        "vdamd_moe_route_small": [P, L, I, I, I, I, I, I, I, P, P, P, P, P, I, P, L, P, I, I, I, I, L, P],
        "vdamd_moe_combine": [P, L, P, L, P, P, P, I, I, I, I, I, P, I, P],
        "vdamd_bias_clamped_glu": [P, L, P, L, P, P, P, I, I, I, I, F, F, I, P],
        "vdamd_moe_topk_grouped": [P, L, P, P, P, I, I, I, I, I, I, I, I, F, I, P],
        "vdamd_mla_attention": [P, L, P, P, P, L, P, P, P, I, P, P, F, I, I, I, I, I, I, I, I, I, I, I, P, P, L, L, P],
        "vdamd_mla_cache_write": [P, L, P, P, P, I, I, I, I, I, I, P],
        "vdamd_mla_prep": [P, P, L, I, I, P, L, L, P, L, P, F, P, P, P, P, P, I, I, I, I, I, I, I, P],
        "vdamd_moe_combine_add_rms_norm": [P, L, P, L, P, P, P, I, I, I, I, I, P, P, F, I, P],
        "vdamd_fp4a16_gemm": [P, L, P, L, P, P, P, P, I, I, I, I, I, I, P],
        "vdamd_fp4_dequant": [P, P, P, P, I, I, I, P],
        "vdamd_fp4a16_gemm_grouped": [P, L, P, L, P, P, L, L, P, P, I, I, I, I, I, P],
        "vdamd_embed_positions": [P, P, P, P, P, I, I, I, I, I, P],
        "vdamd_scalar_norm": [P, P, P, F, I, I, L, I, I, P],
        "vdamd_scalar_norm_residual": [P, P, P, P, P, F, I, I, L, I, I, P],
        "vdamd_poly_norm": [P, P, P, F, I, I, L, I, P],
        "vdamd_conv_norm_cache": [P, L] + [P] * 16 + [I] * 8 + [F, I, P, I, I, P],
        "vdamd_short_conv_act": [P, L, P, L, P, P, P, P, P, P, P] + [I] * 6 + [P, I, P, I, P],
        "vdamd_rotate_norm_cache": [P, P, L, P, I, F, I, F] + [P] * 7 + [I] * 8 + [P],
        "vdamd_window_bias_attention": [P, P, P, P, L, P, P, P, P, P, P, P, P, L, P] + [I] * 10 + [F, F, I, I, I, I, P],
        "vdamd_selective_scan": [P, P, L, P, L, P, P, P, P, P, P, P] + [I] * 7 + [P],
        "vdamd_act_gate_group_norm": [P, P, P, L, P, F, I, I, I, I, P],
        "vdamd_joint_norm_cache": [P, P, L, P, P, F, P, F, I, P, P, P] + [I] * 6 + [P],
        "vdamd_mix_heads": [P, P, P, I, I, I, I, I, P],
        "vdamd_residual_rms": [P, L, P, L, P, L, P, L, P, L, P, L, P, P, P, F, F, I, I, I, I, I, I, F, P],
        "vdamd_gelu_and_mul": [P, P, L, I, I, I, I, P],
        "vdamd_channel_scan": [P, P, L, P, L, P, L, P, L] + [P] * 7 + [I] * 6 + [P],
        "vdamd_block_gates_mfma_ok": [I, I],
        "vdamd_block_gates": [P] * 10 + [L, P, P, P, P, I, I, I, I, P],
        "vdamd_gated_unit_scan": [P, P, P, P, L, P, P, P, P, P, I, I, I, I, P],
        "vdamd_gelu_mul_rows": [P, P, L, P, L, P, I, I, I, I, I, P],
        "vdamd_sigmoid_mul": [P, L, P, L, P, L, F, I, I, I, P],
        "vdamd_gelu": [P, P, L, I, I, P],
        "vdamd_delta_rule_prep": [P, P, P, P, P, L, P, L, P, L, P, P, I, I, I, I, F, I, P],
        "vdamd_delta_rule_rows": [P, P, L, P, L, P, L] + [P] * 6 + [I] * 6 + [F, I, P],
        "vdamd_gated_delta_rule": [P, P, L, I, P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, I, P],
        "vdamd_embed_scaled": [P, P, P, F, I, I, I, I, P],
        "vdamd_layer_norm_to": [P, P, L, P, L, P, P, F, I, I, I, I, I, P],
        "vdamd_gated_rms_norm": [P, L, P, P, P, L, F, I, I, I, F, I, I, I, P],
        "vdamd_clamped_glu": [P, P, L, I, I, F, F, I, P],
        "vdamd_relu_squared": [P, P, L, I, P],
        "vdamd_expert_epilogue": [P, P, P, L, P, P, I, I, P, P, L, I, I, I, P],
        "vdamd_decay_linear_attention": [P, P, L, P, P, P, P, P, I, I, I, I, I, I, I, P],
        "vdamd_channel_decay_attention": [P, P, L, P, P, P, P, P, I, I, I, I, F, I, I, I, P],
        "vdamd_chunk_scan": [P, I, P, L, I, I, I, P, L, P, L, P, P, P, P, P, I, P, P, P, P] + [I] * 9 + [F, F, I, P],
        "vdamd_segment_scan": [P, I, P, L, I, I, I, P, L, P, P, P, P, P, I, I, P, P, P, P] + [I] * 6 + [F, I, P],
        "vdamd_low_rank_decay": [P, P, L, P, P, I, I, I, F, I, P],
        "vdamd_weighted_relu_squared": [P, P, L, P, P, I, I, I, P],
        "vdamd_latent_prep": [P, P, L, L, I, P, L, L, P, L, P, F, P, I, F, P, P, P, P, I, I, I, I, I, I, I, P],
        "vdamd_latent_row_attention": [P, P, P, P, L, P, P, F, I, I, I, I, I, I, P, P, L, I, P],
    }
    for name, argtypes in sigs.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = c_int
    lib.vdamd_chunk_scan_floats.argtypes = [I, I, I]
    lib.vdamd_chunk_scan_floats.restype = c_long
    lib.vdamd_segment_scan_floats.argtypes = [I, I, I]
    lib.vdamd_segment_scan_floats.restype = c_long
    lib.vdamd_decode_workspace_floats.argtypes = [I, I, I]
    lib.vdamd_decode_workspace_floats.restype = c_long
    lib.vdamd_max_splits.restype = c_int
    MAX_SPLITS = int(lib.vdamd_max_splits())
    _LIB = lib
    return lib


# A launch asks for the current stream's handle: 0.2 us of the host by these, 2.7 by an object for the stream (of the 13 that a call of
# one launch then takes: check, allocate, launch)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream() -> int:
    if _raw_stream is None or _current_device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_current_device())


def _check(rc: int, name: str) -> None:
    if rc != 0:
        raise RuntimeError(f"{name} failed with code {rc}")


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}") from None


HEAD_DIMS = (64, 96, 128, 256)


def supports_head_dim(d: int) -> bool:
    """Head sizes the attention kernels are instantiated for (96: Phi-3-mini, 256: Gemma)."""
    return d in HEAD_DIMS


def _half(t: torch.Tensor) -> bool:
    return t.dtype in (torch.bfloat16, torch.float16)


# ------------------------------------------------------------------- norms
def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if not _half(x):
        from . import torch_ref
        return torch_ref.rms_norm(x, weight, eps)
    h = x.shape[-1]
    x2 = x.reshape(-1, h)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    out = torch.empty((x2.shape[0], h), dtype=x.dtype, device=x.device)
    assert weight.numel() == h and weight.dtype == x.dtype and weight.is_contiguous()
    _check(_LIB.vdamd_rms_norm(out.data_ptr(), x2.data_ptr(), None, weight.data_ptr(), eps, x2.shape[0], h,
                               x2.stride(0), h, _dt(x), _stream()), "rms_norm")
    return out.view(x.shape)


def fused_add_rms_norm(x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float,
                       ) -> Tuple[torch.Tensor, torch.Tensor]:
    """In place: ``residual <- x + residual``; ``x <- rms_norm(residual) * w``."""
    if not _half(x):
        from . import torch_ref
        return torch_ref.fused_add_rms_norm(x, residual, weight, eps)
    h = x.shape[-1]
    assert x.dim() == 2 and x.is_contiguous() and residual.is_contiguous() and residual.shape == x.shape
    assert weight.numel() == h and weight.dtype == x.dtype and residual.dtype == x.dtype
    _check(_LIB.vdamd_rms_norm(x.data_ptr(), x.data_ptr(), residual.data_ptr(), weight.data_ptr(), eps,
                               x.shape[0], h, h, h, _dt(x), _stream()), "fused_add_rms_norm")
    return x, residual


def reduce_add_rms_norm(partial: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor,
                        eps: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """``normed = RMSNorm(sum_k partial[k] + residual) * weight`` with ``residual`` updated in place to the
    sum: the K-split slabs ``[ks, T, H]`` (fp32) of the GEMM that fed the norm are reduced by the norm."""
    ks, t, h = partial.shape
    assert partial.dtype == torch.float32 and partial.is_contiguous() and residual.shape == (t, h)
    assert residual.is_contiguous() and _half(residual) and weight.dtype == residual.dtype
    out = torch.empty_like(residual)
    _check(_LIB.vdamd_reduce_add_rms_norm(out.data_ptr(), partial.data_ptr(), ks, residual.data_ptr(),
                                          weight.data_ptr(), float(eps), t, h, h, _dt(residual), _stream()),
           "reduce_add_rms_norm")
    return out, residual


def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    if not _half(x):
        from . import torch_ref
        return torch_ref.layer_norm(x, weight, bias, eps)
    h = x.shape[-1]
    x2 = x.reshape(-1, h).contiguous()
    out = torch.empty_like(x2)
    _check(_LIB.vdamd_layer_norm(out.data_ptr(), x2.data_ptr(), weight.data_ptr(),
                                 None if bias is None else bias.data_ptr(), eps, x2.shape[0], h, _dt(x),
                                 _stream()), "layer_norm")
    return out.view(x.shape)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if not _half(x):
        from . import torch_ref
        return torch_ref.silu_and_mul(x)
    f = x.shape[-1] // 2
    x2 = x.reshape(-1, 2 * f)
    assert x2.is_contiguous()
    out = torch.empty((x2.shape[0], f), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_silu_and_mul(out.data_ptr(), x2.data_ptr(), x2.shape[0], f, _dt(x), _stream()),
           "silu_and_mul")
    return out.view(x.shape[:-1] + (f,))


def embedding(ids: torch.Tensor, weight: torch.Tensor, vocab_start: int = 0,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    if not _half(weight):
        from . import torch_ref
        return torch_ref.embedding(ids, weight, vocab_start, True)
    assert ids.dim() == 1 and weight.is_contiguous()
    if ids.dtype != torch.int32:
        ids = ids.to(torch.int32)
    t, h = ids.shape[0], weight.shape[1]
    if out is None:
        out = torch.empty((t, h), dtype=weight.dtype, device=weight.device)
    assert out.shape == (t, h) and out.dtype == weight.dtype and out.is_contiguous()
    _check(_LIB.vdamd_embedding(out.data_ptr(), ids.data_ptr(), weight.data_ptr(), t, h, vocab_start,
                                weight.shape[0], _dt(weight), _stream()), "embedding")
    return out


# ---------------------------------------------------------- rotary + cache
FP8_KV = torch.float8_e4m3fn


def _kv_args(k_cache: torch.Tensor, kv_scales, hkv: int):
    """(kv_fp8 flag, k_scale pointer, v_scale pointer) for a cache tensor pair."""
    if k_cache.dtype != FP8_KV:
        return 0, None, None
    if kv_scales is None:
        return 1, None, None
    ks, vs = kv_scales
    for t in (ks, vs):
        assert t.dtype == torch.float32 and t.numel() == hkv and t.is_contiguous() and t.device == k_cache.device
    return 1, ks.data_ptr(), vs.data_ptr()


def _check_cache(k_cache: torch.Tensor, v_cache: torch.Tensor, hkv: int, d: int) -> int:
    assert k_cache.dtype == v_cache.dtype
    assert k_cache.dim() == 4 and v_cache.dim() == 6 and k_cache.is_contiguous() and v_cache.is_contiguous()
    nb, h, bs, dd = k_cache.shape
    assert (h, dd) == (hkv, d) and bs % 8 == 0 and tuple(v_cache.shape) == (nb, hkv, d // 16, bs // 8, 16, 8), \
        (k_cache.shape, v_cache.shape)
    assert bs % 8 == 0
    return bs


def rope_and_cache(positions, qkv, cos_sin_cache, k_cache, v_cache, slot_mapping, num_heads, num_kv_heads,
                   head_dim, q_norm_weight=None, k_norm_weight=None, norm_eps: float = 0.0,
                   kv_scales=None) -> torch.Tensor:
    """``q_norm_weight`` / ``k_norm_weight``: RMSNorm each q and k head before rotating (Qwen3)."""
    lanes = head_dim // 16          # the fused q/k norm reduces over an aligned power-of-two lane group
    if not _half(qkv) or head_dim % 16 or (q_norm_weight is not None and (lanes & (lanes - 1) or lanes > 64)):
        from . import torch_ref
        return torch_ref.rope_and_cache(positions, qkv, cos_sin_cache, k_cache, v_cache, slot_mapping,
                                        num_heads, num_kv_heads, head_dim, q_norm_weight, k_norm_weight, norm_eps,
                                        kv_scales)
    if q_norm_weight is not None:
        for w in (q_norm_weight, k_norm_weight):
            assert w.dtype == qkv.dtype and w.numel() == head_dim and w.is_contiguous()
    t = qkv.shape[0]
    qs, ks = num_heads * head_dim, num_kv_heads * head_dim
    assert qkv.dim() == 2 and qkv.shape[1] == qs + 2 * ks and qkv.stride(1) == 1
    assert cos_sin_cache.dtype == torch.float32 and cos_sin_cache.shape[1] == head_dim
    assert positions.dtype == torch.int32 and slot_mapping.dtype == torch.int32
    assert positions.numel() >= t and slot_mapping.numel() >= t
    bs = _check_cache(k_cache, v_cache, num_kv_heads, head_dim)
    st = qkv.stride(0)
    esz = qkv.element_size()
    base = qkv.data_ptr()
    _check(_LIB.vdamd_rope_cache(positions.data_ptr(), base, base + qs * esz, base + (qs + ks) * esz, st, st, st,
                                 cos_sin_cache.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                                 slot_mapping.data_ptr(), t, num_heads, num_kv_heads, head_dim, bs, 0,
                                 None if q_norm_weight is None else q_norm_weight.data_ptr(),
                                 None if k_norm_weight is None else k_norm_weight.data_ptr(), norm_eps,
                                 _dt(qkv), *_kv_args(k_cache, kv_scales, num_kv_heads), _stream()), "rope_and_cache")
    return qkv[:, :qs]


def rope_and_cache_partials(positions, slabs, dtype, cos_sin_cache, k_cache, v_cache, slot_mapping, num_heads,
                            num_kv_heads, head_dim, q_norm_weight=None, k_norm_weight=None, norm_eps: float = 0.0,
                            kv_scales=None) -> torch.Tensor:
    """``rope_and_cache`` whose packed ``qkv`` arrives as the fp32 K-split slabs ``[ks, T, (Hq + 2 Hkv) D]`` of
    the projection (summed here, rounded to ``dtype`` first as the GEMM's own reduction would); returns the
    rotated ``q [T, Hq D]`` in a buffer of its own."""
    ks, t, n = slabs.shape
    qs = num_heads * head_dim
    lanes = head_dim // 16
    assert slabs.dtype == torch.float32 and slabs.is_contiguous() and n == qs + 2 * num_kv_heads * head_dim
    assert head_dim % 16 == 0 and dtype in (torch.bfloat16, torch.float16)
    assert q_norm_weight is None or (lanes & (lanes - 1) == 0 and lanes <= 64)
    if q_norm_weight is not None:
        for w in (q_norm_weight, k_norm_weight):
            assert w.dtype == dtype and w.numel() == head_dim and w.is_contiguous()
    assert cos_sin_cache.dtype == torch.float32 and cos_sin_cache.shape[1] == head_dim
    assert positions.dtype == torch.int32 and slot_mapping.dtype == torch.int32
    assert positions.numel() >= t and slot_mapping.numel() >= t
    bs = _check_cache(k_cache, v_cache, num_kv_heads, head_dim)
    q = torch.empty((t, qs), dtype=dtype, device=slabs.device)
    _check(_LIB.vdamd_rope_cache_slabs(positions.data_ptr(), slabs.data_ptr(), ks, q.data_ptr(), qs,
                                       cos_sin_cache.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                                       slot_mapping.data_ptr(), t, num_heads, num_kv_heads, head_dim, bs,
                                       None if q_norm_weight is None else q_norm_weight.data_ptr(),
                                       None if k_norm_weight is None else k_norm_weight.data_ptr(), norm_eps,
                                       _DT[dtype],
                                       *_kv_args(k_cache, kv_scales, num_kv_heads), _stream()),
           "rope_and_cache_partials")
    return q


def rotary_embedding(positions, q, k, cos_sin_cache, head_dim) -> None:
    if not _half(q):
        from . import torch_ref
        return torch_ref.rotary_embedding(positions, q, k, cos_sin_cache, head_dim)
    t = q.shape[0]
    assert q.stride(-1) == 1 and k.stride(-1) == 1 and q.dim() == 2 and k.dim() == 2
    assert positions.dtype == torch.int32 and cos_sin_cache.dtype == torch.float32
    _check(_LIB.vdamd_rope_cache(positions.data_ptr(), q.data_ptr(), k.data_ptr(), None, q.stride(0),
                                 k.stride(0), 0, cos_sin_cache.data_ptr(), None, None, None, t,
                                 q.shape[1] // head_dim, k.shape[1] // head_dim, head_dim, 16, 1, None, None, 0.0,
                                 _dt(q), 0, None, None, _stream()), "rotary_embedding")


def reshape_and_cache(k, v, k_cache, v_cache, slot_mapping, kv_scales=None) -> None:
    if not _half(k):
        from . import torch_ref
        return torch_ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping, kv_scales)
    t, hkv, d = k.shape
    assert k.stride(2) == 1 and v.stride(2) == 1 and k.stride(1) == d and v.stride(1) == d
    assert slot_mapping.dtype == torch.int32 and slot_mapping.numel() >= t
    bs = _check_cache(k_cache, v_cache, hkv, d)
    _check(_LIB.vdamd_rope_cache(None, None, k.data_ptr(), v.data_ptr(), 0, k.stride(0), v.stride(0), None,
                                 k_cache.data_ptr(), v_cache.data_ptr(), slot_mapping.data_ptr(), t, 0, hkv, d,
                                 bs, 2, None, None, 0.0, _dt(k), *_kv_args(k_cache, kv_scales, hkv), _stream()),
           "reshape_and_cache")


# ---------------------------------------------------------------- attention
def decode_workspace_floats(max_bs: int, num_heads: int, head_dim: int, num_kv_heads: int = 1,
                            max_seq_len: int = 1 << 30) -> int:
    """Floats of split-KV scratch that cover every batch size up to ``max_bs``
    (splits shrink as the batch grows, so this is far below max_bs * MAX_SPLITS)."""
    worst = max(b * choose_num_splits(b, num_kv_heads, max_seq_len) for b in range(1, max(1, max_bs) + 1))
    return worst * num_heads * (head_dim + 2)


def choose_num_splits(batch: int, num_kv_heads: int, max_seq_len: int, captured: bool = True) -> int:
    """KV splits of a decode step, ``captured`` in a graph or launched from Python.

    The four waves of a workgroup take the keys 32 at a time in turn, so a long context on few workgroups is a serial chain:
    where the (sequence, KV head) pairs leave room for three splits each, as many splits of at least 64 keys as make 512
    workgroups.  One sequence of 8 heads over 800 keys takes 12.5 us whole and 8.5 in 12 splits, over 2000 keys 14.2 in 3 and 8.9
    in 31.  A merge costs what that saves below about 512 keys, and later the more workgroups there are (64 of them over 520 keys:
    9.3 whole, 9.0 in 8; 160 over 800 keys 17.5 and 18.5, over 1400 keys 26 in 2 and 24 in 4).  With a workgroup for most CUs a
    split only adds the partial sums (192 over 800 keys: 18 whole, 20 in 3; 32 x 8 heads over 1000 keys: 22.5 whole, 25.9 in 2)
    unless contexts are long enough to end unevenly (32 x 8 heads over about 9000 keys: 354 whole, 311 in 2): splits of at least
    512 keys, and as many as make 512 workgroups or more (20 x 8 heads over 4000 keys: 62.8 in 3, 58.4 in 4).
    Outside a graph a second launch costs the host 4.5 us (13.5 and 18.0 us a call), more than it saves below 1024 keys."""
    wgs = max(1, batch * num_kv_heads)
    long = min((512 + wgs - 1) // wgs, max_seq_len // 512)
    if 512 // wgs >= 3:
        whole = 512 + 3 * wgs if captured else 1024
        long = 1 if max_seq_len < whole else max(long, min(512 // wgs, max_seq_len // 64))
    return max(1, min(MAX_SPLITS, long))


def _per_head(t: Optional[torch.Tensor], hq: int, q: torch.Tensor):
    """Pointer of an optional fp32 ``[Hq]`` vector (attention sinks, ALiBi slopes)."""
    if t is None:
        return None
    assert t.dtype == torch.float32 and t.numel() == hq and t.is_contiguous() and t.device == q.device
    return t.data_ptr()


# decode attention reads more than this past the chip's caches (256 MB of them on the memory's side)
DECODE_ONCE_BYTES = 208 << 20


def decode_reads_once(batch: int, heads: int, num_kv_heads: int, head_dim: int, keys: int) -> bool:
    """Whether a decode step over a 16-bit cache may read keys and values past the caches: if every row saw ``keys`` of them they
    would be too many to be kept, and each is read by one workgroup only (with two tiles of query heads to a key head, 64 over
    2 of 128, 48 rows of about 9000 keys, 141 us through the caches and 174 past them; with five, 71 over 1 of 64, 153 and 236).
    What the rows do see, and which pages several of them share, the kernel asks where it runs: ``keys`` is a bound, in a graph
    a loose one.  Several caches in turn, us (cached / past them / asking first): 48 rows of about 9000 keys, 32 heads over 8 of
    128, 318 / 302 / 304, 256 of 400 86 / 79 / 78, with three quarters of the pages shared 210 / 241 / 219 and, 128 rows of
    3000, 186 / 210 / 186; 16 rows of 1000, which four caches hold, under a bound of 32768 18.2 / 20.6 / 18.5."""
    if -(-heads // num_kv_heads) > 16 or head_dim > 128:
        return False
    return batch * keys * num_kv_heads * head_dim * 4 >= DECODE_ONCE_BYTES


def paged_attention_decode(q, k_cache, v_cache, block_table, seq_lens, scale, max_seq_len=0, out=None,
                           workspace=None, num_splits: Optional[int] = None, kv_scales=None,
                           window: int = 0, softcap: float = 0.0, sinks=None, alibi_slopes=None) -> torch.Tensor:
    """``window > 0``: sliding-window attention, the query sees its last ``window`` keys only.
    ``softcap > 0``: scores become ``softcap * tanh(score / softcap)`` before the softmax (Gemma-2).
    ``sinks [Hq]`` (fp32): one extra score per query head that only enters the softmax's denominator
    (attention sinks).  ``alibi_slopes [Hq]`` (fp32): key ``k`` gets ``slope * (k - query position)`` added."""
    b, hq, d = q.shape
    hkv = k_cache.shape[1]
    bs = _check_cache(k_cache, v_cache, hkv, d)
    assert q.stride(2) == 1 and q.stride(1) == d and hq % hkv == 0
    assert block_table.dtype == torch.int32 and seq_lens.dtype == torch.int32
    assert block_table.shape[0] >= b and seq_lens.numel() >= b and block_table.stride(1) == 1
    if max_seq_len <= 0:
        max_seq_len = block_table.shape[1] * bs
    assert max_seq_len <= block_table.shape[1] * bs, "block table narrower than max_seq_len"
    if out is None:
        out = torch.empty((b, hq, d), dtype=q.dtype, device=q.device)
    assert out.is_contiguous() and out.shape == (b, hq, d)
    keys = min(max_seq_len, window) if window > 0 else max_seq_len
    if num_splits is None:
        # (whole up to 512 keys and the same from 1024 on: asking costs 0.4 us)
        num_splits = choose_num_splits(b, hkv, keys, keys >= 1024 or keys > 512 and torch.cuda.is_current_stream_capturing())
    ws_ptr = None
    assert 0 <= num_splits <= MAX_SPLITS       # 0 = the one-wave-per-sequence kernel
    if num_splits > 1:
        need = b * hq * num_splits * (d + 2)
        if workspace is None or workspace.numel() < need:
            workspace = torch.empty(need, dtype=torch.float32, device=q.device)
        ws_ptr = workspace.data_ptr()
    kv = _kv_args(k_cache, kv_scales, hkv)
    past = max(1, DECODE_ONCE_BYTES) if kv[0] == 0 and num_splits and decode_reads_once(b, hq, hkv, d, keys) else 0
    _check(_LIB.vdamd_paged_attention_decode(
        out.data_ptr(), ws_ptr, q.data_ptr(), q.stride(0), k_cache.data_ptr(), v_cache.data_ptr(),
        block_table.data_ptr(), block_table.stride(0), seq_lens.data_ptr(), float(scale), b, hq, hkv, d, bs,
        num_splits, hq * d, _dt(q), *kv, int(window), float(softcap),
        _per_head(sinks, hq, q), _per_head(alibi_slopes, hq, q), past, _stream()), "paged_attention_decode")
    return out


def paged_attention_prefill(q, k_cache, v_cache, block_table, query_start_loc, seq_lens, scale,
                            max_query_len=0, max_seq_len=0, out=None, kv_scales=None, window: int = 0,
                            softcap: float = 0.0, sinks=None, alibi_slopes=None) -> torch.Tensor:
    t, hq, d = q.shape
    hkv = k_cache.shape[1]
    bs = _check_cache(k_cache, v_cache, hkv, d)
    nseq = seq_lens.numel()
    assert q.stride(2) == 1 and q.stride(1) == d and hq % hkv == 0
    assert block_table.dtype == torch.int32 and seq_lens.dtype == torch.int32
    assert query_start_loc.dtype == torch.int32 and query_start_loc.numel() == nseq + 1
    assert block_table.shape[0] >= nseq and block_table.stride(1) == 1
    if max_query_len <= 0:
        max_query_len = t
    if max_seq_len > 0:
        assert max_seq_len <= block_table.shape[1] * bs, "block table narrower than max_seq_len"
    if out is None:
        out = torch.empty((t, hq, d), dtype=q.dtype, device=q.device)
    assert out.is_contiguous() and out.shape == (t, hq, d)
    _check(_LIB.vdamd_paged_attention_prefill(
        out.data_ptr(), q.data_ptr(), q.stride(0), k_cache.data_ptr(), v_cache.data_ptr(),
        block_table.data_ptr(), block_table.stride(0), query_start_loc.data_ptr(), seq_lens.data_ptr(),
        float(scale), nseq, max_query_len, hq, hkv, d, bs, hq * d, _dt(q), *_kv_args(k_cache, kv_scales, hkv),
        int(window), float(softcap), _per_head(sinks, hq, q), _per_head(alibi_slopes, hq, q), _stream()),
        "paged_attention_prefill")
    return out


# ----------------------------------------------------------------- sampling
def argmax(logits: torch.Tensor) -> torch.Tensor:
    assert logits.dim() == 2 and logits.stride(1) == 1
    b, v = logits.shape
    out = torch.empty(b, dtype=torch.int32, device=logits.device)
    _check(_LIB.vdamd_argmax(out.data_ptr(), logits.data_ptr(), b, v, logits.stride(0), _dt(logits),
                             _stream()), "argmax")
    return out


def sample(logits, temperature, top_k, top_p, min_p, uniform) -> torch.Tensor:
    assert logits.dim() == 2 and logits.stride(1) == 1
    b, v = logits.shape
    for t, dt in ((temperature, torch.float32), (top_k, torch.int32), (top_p, torch.float32),
                  (min_p, torch.float32), (uniform, torch.float32)):
        assert t.dtype == dt and t.numel() == b and t.is_contiguous() and t.is_cuda
    out = torch.empty(b, dtype=torch.int32, device=logits.device)
    _check(_LIB.vdamd_sample(out.data_ptr(), logits.data_ptr(), b, v, logits.stride(0), temperature.data_ptr(),
                             top_k.data_ptr(), top_p.data_ptr(), min_p.data_ptr(), uniform.data_ptr(),
                             _dt(logits), _stream()), "sample")
    return out


# ------------------------------------------------------------ W4A16 linears
W4_MAX_FUSED_M = int(os.environ.get("VDAMD_W4_MAX_FUSED_M", "256"))


def _w4_dims(qw: torch.Tensor, sz: torch.Tensor) -> Tuple[int, int, int]:
    assert qw.dim() == 4 and qw.shape[2:] == (64, 4) and qw.dtype == torch.int32 and qw.is_contiguous()
    n, k = qw.shape[0] * 16, qw.shape[1] * 128
    assert sz.dim() == 4 and sz.shape[0] == qw.shape[0] and sz.shape[2:] == (16, 2) and sz.is_contiguous()
    g = k // sz.shape[1]
    assert g * sz.shape[1] == k and g % 128 == 0, (k, sz.shape)
    return n, k, g


def w4_choose_variant(m: int, n: int, k: int) -> int:
    """0: waves split K, x from L2 (finest tiling; best for one row tile);
    1: waves split N and share x through LDS (batches above 16 rows, when
    there are enough 256-row workgroups to go round)."""
    override = os.environ.get("VDAMD_W4_VARIANT")
    if override is not None:
        return int(override)
    if m <= 16 or (m <= 32 and n < 32768):      # measured inside a captured graph on 70B / 480B projections
        return 0
    wgs = ((n // 16 + 15) // 16) * max(1, (k // 128) // 4)
    return 1 if wgs >= 128 else 0


def w4_choose_ksplit(m: int, n: int, k: int, variant: int = 0) -> int:
    """Split K until ~2-3 workgroups per CU exist (variant 0: 64 rows per
    workgroup, at least two 128-column blocks per wave; variant 1: 256 output
    rows per workgroup up to 64 batch rows, 128 above (row chunks of <= 128),
    at least four blocks per workgroup)."""
    if variant == 1:
        if m > 64:
            base = ((n // 16 + 7) // 8) * ((m + 127) // 128)
        else:
            base = (n // 16 + 15) // 16
        return max(1, min((512 + base - 1) // base, (k // 128) // 4))
    mt = min(4, (m + 15) // 16)
    mz = (m + 16 * mt - 1) // (16 * mt)
    base = ((n // 16 + 3) // 4) * mz
    ks = max(1, min((512 + base - 1) // base, (k // 128) // 8))
    return 1 << (ks.bit_length() - 1)       # power-of-two splits measured at or next to the optimum; 3 and 6 are not


def w4_dequant(qw: torch.Tensor, sz: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    n, k, g = _w4_dims(qw, sz)
    if out is None:
        out = torch.empty((n, k), dtype=sz.dtype, device=qw.device)
    assert out.is_contiguous() and out.numel() >= n * k and out.dtype == sz.dtype
    _check(_LIB.vdamd_w4_dequant(out.data_ptr(), qw.data_ptr(), sz.data_ptr(), n, k, g, _dt(sz), _stream()),
           "w4_dequant")
    return out[:n * k].view(n, k) if out.dim() == 1 else out


def w4a16_gemm(x: torch.Tensor, qw: torch.Tensor, sz: torch.Tensor, variant: Optional[int] = None,
               ksplit: Optional[int] = None, partials: bool = False) -> Optional[torch.Tensor]:
    """``x [M, K]`` (bf16/fp16, rows 16-byte aligned) times the packed weights.  ``partials``: the fp32
    K-split slabs ``[ksplit, M, N]`` instead of their sum, for a consumer that adds them up while it
    reads them; None when the shape runs unsplit."""
    n, k, g = _w4_dims(qw, sz)
    assert x.dim() == 2 and x.shape[1] == k and x.dtype == sz.dtype and x.stride(1) == 1
    assert x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
    m = x.shape[0]
    if variant is None:
        variant = w4_choose_variant(m, n, k)
    if ksplit is None:
        ksplit = w4_choose_ksplit(m, n, k, variant)
    if partials and (ksplit <= 1 or m == 0):
        return None
    out = None if partials else torch.empty((m, n), dtype=x.dtype, device=x.device)
    if m == 0:
        return out
    assert 1 <= ksplit <= k // 128
    partial = torch.empty((ksplit, m, n), dtype=torch.float32, device=x.device) if ksplit > 1 else None
    _check(_LIB.vdamd_w4a16_gemm(None if out is None else out.data_ptr(), n, x.data_ptr(), x.stride(0), qw.data_ptr(),
                                 sz.data_ptr(), None if partial is None else partial.data_ptr(), m, n, k, g, ksplit,
                                 variant, _dt(x), _stream()), "w4a16_gemm")
    return partial if partials else out


# ------------------------------------------------------------ NVFP4 linears
def _fp4_dims(qw: torch.Tensor, fs: torch.Tensor, alpha: Optional[torch.Tensor]) -> Tuple[int, int]:
    assert qw.dim() == 4 and qw.shape[2:] == (64, 4) and qw.dtype == torch.int32 and qw.is_contiguous()
    assert fs.shape == qw.shape[:2] + (64,) and fs.dtype == torch.int32 and fs.is_contiguous()
    n, k = qw.shape[0] * 16, qw.shape[1] * 128
    if alpha is not None:
        assert alpha.dtype == torch.float32 and alpha.numel() == n and alpha.is_contiguous()
    return n, k


def fp4_dequant(qw: torch.Tensor, fs: torch.Tensor, alpha: Optional[torch.Tensor], dtype: torch.dtype,
                out: Optional[torch.Tensor] = None) -> torch.Tensor:
    n, k = _fp4_dims(qw, fs, alpha)
    if out is None:
        out = torch.empty((n, k), dtype=dtype, device=qw.device)
    assert out.is_contiguous() and out.numel() >= n * k and out.dtype == dtype
    _check(_LIB.vdamd_fp4_dequant(out.data_ptr(), qw.data_ptr(), fs.data_ptr(),
                                  None if alpha is None else alpha.data_ptr(), n, k, _DT[dtype], _stream()),
           "fp4_dequant")
    return out[:n * k].view(n, k) if out.dim() == 1 else out


def fp4a16_gemm(x: torch.Tensor, qw: torch.Tensor, fs: torch.Tensor, alpha: Optional[torch.Tensor] = None,
                variant: Optional[int] = None, ksplit: Optional[int] = None) -> torch.Tensor:
    """``x [M, K]`` (bf16/fp16) times NVFP4 weights (``ops.quant.pack_fp4``), ``alpha [N]`` fp32 per-row scale."""
    n, k = _fp4_dims(qw, fs, alpha)
    assert x.dim() == 2 and x.shape[1] == k and _half(x) and x.stride(1) == 1
    assert x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
    m = x.shape[0]
    out = torch.empty((m, n), dtype=x.dtype, device=x.device)
    if m == 0:
        return out
    if variant is None:
        variant = w4_choose_variant(m, n, k)
    if ksplit is None:
        ksplit = w4_choose_ksplit(m, n, k, variant)
    assert 1 <= ksplit <= k // 128
    partial = torch.empty(ksplit * m * n, dtype=torch.float32, device=x.device) if ksplit > 1 else None
    _check(_LIB.vdamd_fp4a16_gemm(out.data_ptr(), n, x.data_ptr(), x.stride(0), qw.data_ptr(), fs.data_ptr(),
                                  None if alpha is None else alpha.data_ptr(),
                                  None if partial is None else partial.data_ptr(), m, n, k, ksplit, variant,
                                  _dt(x), _stream()), "fp4a16_gemm")
    return out


# ---------------------------------------------------------- skinny bf16 GEMM
SKINNY_MAX_M = 128


def skinny_supported(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.dim() == 2 and w.dim() == 2 and 0 < x.shape[0] <= SKINNY_MAX_M and x.dtype == w.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and x.shape[1] == w.shape[1]
            and w.shape[1] % 128 == 0 and w.shape[0] % 16 == 0 and x.stride(1) == 1 and w.stride(1) == 1
            and x.stride(0) % 8 == 0 and w.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
            and w.data_ptr() % 16 == 0)


def skinny_choose(m: int, n: int, k: int) -> Tuple[int, int]:
    """``(ntw, ksplit)``: output tiles per wave and K split.  Fewer tiles per
    wave when N alone cannot fill the chip; then K is split until there are
    about two workgroups per CU, keeping >= 4 column blocks per workgroup.
    Long-K shapes (the down projection) and wide short-K ones (an 8B-class
    gate_up) use the measured optimum."""
    tiles = n // 16
    if k >= 2 * n and k >= 8192:
        if tiles <= 256:                      # e.g. 4096 x 14336: one tile per wave, 64 workgroups x 8
            return 1, max(1, min(8, (k // 128) // 4))
        ntw = 1 if m <= 32 else (4 if m <= 64 else 2)
        wgs = (tiles + 4 * ntw - 1) // (4 * ntw)
        return ntw, max(1, min(4 if m <= 32 else 8, (1024 + wgs - 1) // wgs, (k // 128) // 4))
    if m <= 16 and n >= 16384 and k <= 4096:
        return 2, max(1, min(4, (k // 128) // 4))
    ntw = 4 if m <= 64 else 2
    while ntw > 1 and (tiles + 4 * ntw - 1) // (4 * ntw) < 512:
        ntw //= 2
    wgs = (tiles + 4 * ntw - 1) // (4 * ntw)
    ksplit = max(1, min((512 + wgs - 1) // wgs, (k // 128) // 4))
    return ntw, ksplit


def skinny_profitable(m: int, n: int, k: int) -> bool:
    """Where this kernel beats the library GEMM on MI355X (measured in captured
    graphs, benchmarks/skinny_gemm_bench.py): long reductions into a narrow
    output, for which the library's short-batch kernels reach only 1.6-4.8 TB/s
    (from 24 rows up when the output is 4096 wide or less - below that the
    two are level), very wide outputs over a short reduction at <= 16 rows, and
    4096-square projections at <= 16 rows."""
    if m > SKINNY_MAX_M:
        return False
    if k >= 2 * n and k >= 8192:
        return m >= 24 or n > 4096
    if m <= 16 and 2048 <= n <= 4096 and 4096 <= k < 8192:      # a square 4096 projection: 11.2 vs 12.5 us at one row
        return True
    return m <= 16 and n >= 16384 and k <= 4096


def skinny_gemm(x: torch.Tensor, w: torch.Tensor, ntw: Optional[int] = None, ksplit: Optional[int] = None,
                out: Optional[torch.Tensor] = None, silu_mul: bool = False) -> torch.Tensor:
    """``x [M<=128, K] @ w [N, K]^T`` streaming ``w`` once at HBM speed.  ``silu_mul``: ``x`` is
    ``[M, 2K] = [gate | up]`` and the left operand is ``silu(gate) * up``, formed inside the kernel."""
    up_off = 0
    if silu_mul:
        assert x.dim() == 2 and x.shape[1] == 2 * w.shape[1] and x.stride(1) == 1
        up_off = w.shape[1]
        x = x[:, :up_off]                      # the gate half; the kernel finds the up half up_off further on
    assert skinny_supported(x, w), (x.shape, x.stride(), w.shape, w.stride(), x.dtype)
    m, k = x.shape
    n = w.shape[0]
    a, b = skinny_choose(m, n, k)
    ntw = a if ntw is None else ntw
    ksplit = b if ksplit is None else ksplit
    assert 1 <= ksplit <= k // 128
    if out is None:
        out = torch.empty((m, n), dtype=x.dtype, device=x.device)
    assert out.shape == (m, n) and out.dtype == x.dtype and out.is_contiguous() and out.data_ptr() % 16 == 0
    partial = torch.empty(ksplit * m * n, dtype=torch.float32, device=x.device) if ksplit > 1 else None
    _check(_LIB.vdamd_skinny_gemm(out.data_ptr(), n, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                                  None if partial is None else partial.data_ptr(), m, n, k, ksplit, ntw,
                                  _dt(x), up_off, _stream()), "skinny_gemm")
    return out


def skinny_gemm_partials(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """``skinny_gemm`` without its reduction: the fp32 partial sums ``[ksplit, M, N]`` of ``x @ w^T``, for a
    consumer that adds them up while it loads them (the decode routing kernel).  None when the shape is
    not split over K (there is then nothing to save) or not one the kernel takes."""
    if not skinny_supported(x, w):
        return None
    m, k = x.shape
    n = w.shape[0]
    ntw, ksplit = skinny_choose(m, n, k)
    if ksplit <= 1:
        return None
    partial = torch.empty((ksplit, m, n), dtype=torch.float32, device=x.device)
    _check(_LIB.vdamd_skinny_gemm(None, n, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), partial.data_ptr(),
                                  m, n, k, ksplit, ntw, _dt(x), 0, _stream()), "skinny_gemm (partial sums)")
    return partial


# ------------------------------------------- weight-streaming GEMM, M <= 16
STREAM_MAX_M = 16
EPI_NONE, EPI_RESIDUAL, EPI_SILU_MUL = 0, 1, 2


def stream_supported(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.dim() == 2 and w.dim() == 2 and 0 < x.shape[0] <= STREAM_MAX_M and x.dtype == w.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and x.shape[1] == w.shape[1]
            and w.shape[1] % 128 == 0 and w.shape[0] % 16 == 0 and x.stride(1) == 1 and w.stride(1) == 1
            and x.stride(0) % 8 == 0 and w.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
            and w.data_ptr() % 16 == 0)


STREAM_WIRED_MAX_M = 8


def stream_profitable(m: int, n: int, k: int) -> bool:
    """Up to 8 rows into a very wide output over a reduction of 2048 to 4095; longer ones are ``mid_gemm``'s (28672 x 4096 by one
    row 47 us here, 41 there), narrow outputs (a TP=8 shard) the library's.  With SiLU * up, us at 1 / 8 rows, here, by
    ``mid_gemm`` and by library and activation kernel: 28672 x 2048 28 / 31, 23 / 23, 42 / 41; 49152 x 3072 55 / 57, 60 / 60,
    74 / 74; 37888 x 3584 51 / 54, 58 / 60, 65 / 69; 30720 x 3840 48 / 53, 41 / 42, 60 / 60: ahead of ``mid_gemm`` only where
    that one's last round is nearly empty."""
    return 0 < m <= STREAM_WIRED_MAX_M and n >= MID_SILU_MIN_N and 2048 <= k < MID_SILU_MIN_K


def stream_choose(n: int, k: int, silu: bool = False) -> Tuple[int, int, int]:
    """``(ntw, ksplit, depth)``.  One output tile per workgroup until N alone gives several
    workgroups per CU; K is split across workgroups only when even that leaves CUs idle."""
    tiles = n // 16
    ntw = 2 if (silu or tiles >= 4096) else 1
    wgs = tiles // ntw
    ksplit = 1
    while wgs * ksplit < 1024 and (k // 128) // (ksplit * 2) >= 8:
        ksplit *= 2
    return ntw, ksplit, 3


def stream_gemm(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None,
                residual: Optional[torch.Tensor] = None, silu_mul: bool = False, ntw: Optional[int] = None,
                ksplit: Optional[int] = None, depth: Optional[int] = None, nt: bool = False) -> torch.Tensor:
    """``x [M<=16, K] @ w [N, K]^T`` reading ``w`` once at HBM speed.  ``residual [M, N]`` is added in
    the epilogue; ``silu_mul`` treats ``w`` as ``[gate ; up]`` and returns ``silu(gate) * up`` (``N/2`` wide)."""
    assert stream_supported(x, w), (x.shape, x.stride(), w.shape, w.stride(), x.dtype)
    assert not (silu_mul and residual is not None)
    m, k = x.shape
    n = w.shape[0]
    a, b, c = stream_choose(n, k, silu_mul)
    ntw = a if ntw is None else ntw
    ksplit = b if ksplit is None else ksplit
    depth = c if depth is None else depth
    n_out = n // 2 if silu_mul else n
    if out is None:
        out = torch.empty((m, n_out), dtype=x.dtype, device=x.device)
    assert out.shape == (m, n_out) and out.dtype == x.dtype and out.stride(1) == 1 and out.data_ptr() % 8 == 0
    epi = EPI_SILU_MUL if silu_mul else (EPI_RESIDUAL if residual is not None else EPI_NONE)
    if residual is not None:
        assert residual.shape == (m, n) and residual.dtype == x.dtype and residual.stride(1) == 1
    partial = torch.empty(ksplit * m * n, dtype=torch.float32, device=x.device) if ksplit > 1 else None
    _check(_LIB.vdamd_stream_gemm(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(),
                                  w.stride(0), None if partial is None else partial.data_ptr(),
                                  None if residual is None else residual.data_ptr(),
                                  0 if residual is None else residual.stride(0), m, n, k, ksplit, ntw, depth,
                                  int(nt), epi, _dt(x), _stream()), "stream_gemm")
    return out


# ---------------------------------------- split-K LDS-DMA GEMM, 1 <= M <= 1280
MID_MAX_M = 1280


def mid_supported(x: torch.Tensor, w: torch.Tensor, silu_mul: bool = False) -> bool:
    return (x.dim() == 2 and w.dim() == 2 and 0 < x.shape[0] <= MID_MAX_M and x.dtype == w.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and x.shape[1] == w.shape[1]
            and w.shape[1] % 64 == 0 and w.shape[0] % (32 if silu_mul else 16) == 0 and x.stride(1) == 1 and w.stride(1) == 1
            and x.stride(0) % 8 == 0 and w.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
            and w.data_ptr() % 16 == 0 and max(x.stride(0), w.stride(0)) < (1 << 22)
            and (not silu_mul or w.shape[0] * w.stride(0) * 2 < (1 << 32) - 64))


def mid_out_ok(out: Optional[torch.Tensor], x: torch.Tensor, n: int) -> bool:
    """Whether the kernel can write its rows into ``out`` (the library takes any other strides and places)."""
    return out is None or (out.shape == (x.shape[0], n) and out.dtype == x.dtype and out.stride(1) == 1
                           and out.stride(0) % 4 == 0 and out.data_ptr() % 8 == 0)


def mid_bias_ok(bias: torch.Tensor, x: torch.Tensor, w: torch.Tensor) -> bool:
    return (bias.shape == w.shape[:1] and bias.dtype == x.dtype and bias.is_cuda and bias.is_contiguous()
            and bias.data_ptr() % 8 == 0)


# workgroup tile: us of a launch apart from its K tiles, us of one 64-deep K tile of a workgroup, workgroups that run at once,
# TB/s of W that those reach.  Fitted by least squares; against 4294 timings of 21 weight shapes (8 MB to 2.1 GB) at 1 to 512 rows
# and every split 8.4 % off in the mean, the chosen tile and split 3.3 % above the fastest in the mean, 40 % at most (8192 x
# 1024 at 256 rows and above; profiles/mid_gemm_tiles_mi355x.txt, from benchmarks/stream_gemm_sweep.py --model).  Tiles of 192 rows,
# for 129 to 192, 257 to 384 and 513 to 576: of the 432 products of 130 to 1280 rows there that this kernel takes, the choice is 1.8 %
# above the fastest in the mean, 15 % at most.
_MID_TILES = {(256, 256): (7.1, 1.21, 256, 5.9), (256, 128): (5.4, 0.76, 256, 4.8), (192, 256): (6.8, 0.8, 256, 5.9),
              (192, 128): (4.0, 0.75, 256, 5.4), (128, 256): (6.5, 0.89, 256, 5.9),
              (128, 128): (4.4, 0.59, 256, 5.9), (64, 128): (4.0, 0.45, 512, 5.9)}
# K-split counts the choice is made from (VDAMD_MID_KSPLITS=1,2,4,8,16 restricts it, for A/B measurements)
_MID_KSPLITS = tuple(int(v) for v in os.environ.get("VDAMD_MID_KSPLITS", "1,2,3,4,5,6,7,8,12,16").split(","))
if os.environ.get("VDAMD_MID_GEMM_VARIANT", "-1") != "-1":
    logger.warning("VDAMD_MID_GEMM_VARIANT has no effect: what it chose between is one kernel now")


def _mid_blocks(m: int, n: int, bm: int, bn: int, ksplit: int) -> int:
    return -(-n // bn) * ksplit * -(-m // bm)


def _mid_estimate(m: int, n: int, k: int, bm: int, bn: int, ksplit: int, reduced: bool) -> float:
    """Modelled run time in us: rounds of workgroups x K tiles x time per tile, at least that of reading its part of W, plus
    the fp32 slabs, written and read again, and the launch that sums them up."""
    fixed, tile_us, slots, tbs = _MID_TILES[(bm, bn)]
    rounds, left = divmod(_mid_blocks(m, n, bm, bn, ksplit), slots)
    read_us = bn * 128 / (tbs * 1e6)       # per K tile and workgroup, at the full rate once most CUs read
    tile = rounds * max(tile_us, read_us * slots / min(1.0, 0.5 + slots / 440))
    if left:
        tile += max(tile_us, read_us * left / min(1.0, 0.5 + left / 440))
    if rounds + (left > 0) > 1:            # a CU's one workgroup fills and drains its ring in every round
        tile *= 1.25 if bn == 128 and slots == 256 else 1.1
    slabs = ((3.0 if reduced else 0.0) + ksplit * m * n * 4 * 0.4e-6) if ksplit > 1 else 0.0
    if bm == 192 and ksplit == 16:         # (2048 x 12288 at 160 rows 25.7 us in 16 splits, 23.2 in 12)
        slabs += 1.5
    total = fixed + k / 64 / ksplit * tile + slabs
    # (K in slices of a multiple of 16 KB, few rows in the last of several tiles: 257 rows of 8192 x 16384 in tiles of 192 x 128 and
    # halves of K 156 us, 384 rows 112, 257 in tiles of 192 x 256 and quarters 107)
    if bn == 128 and ksplit > 1 and k // ksplit % 8192 == 0 and m > bm and (m - 1) % bm < bm // 2:
        total *= 1.4
    return total


# The rules below are functions of whole numbers alone, asked several times for every product of a step that runs outside a
# graph: their answers are kept (by shape, the last 4096 of them; 50 to 150 us a question, as much as a product takes, against 0.1)
@functools.lru_cache(maxsize=4096)
def mid_choose(m: int, n: int, k: int, reduced: bool = True) -> Tuple[int, int, int]:
    """``(bm, bn, ksplit)`` with the smallest modelled time.  The row tile covers all of M up to 256
    (W is then read from HBM once), above that whatever pads the last one least may be the faster (557 rows of 4096 x 14336: 75 us in
    three tiles of 192, 88 of 256); splitting K buys parallelism and costs slab traffic."""
    best = None
    for (bm, bn) in _MID_TILES:
        if bm < (min(m, 256) if m <= 256 else 192 if m <= 512 else 128) or (bm > 64 and bm >= 4 * m):
            continue
        # (counts that are not powers of two as well: a 70B qkv projection's 80 column tiles fill 240 of the
        # 256 CUs at 3, 160 at 2)
        for ksplit in _MID_KSPLITS:
            if ksplit > 1 and k // 64 // ksplit < (4 if ksplit <= 8 else 8):
                break
            e = _mid_estimate(m, n, k, bm, bn, ksplit, reduced)
            if best is None or e < best[0]:
                best = (e, bm, bn, ksplit)
    return best[1], best[2], best[3]


@functools.lru_cache(maxsize=4096)
def mid_silu_tile(m: int, n: int, k: int) -> Tuple[int, int]:
    """The tile of the unsplit form with the activation in its epilogue."""
    return min((t for t in _MID_TILES if t[0] >= m or t[0] == 256), key=lambda t: _mid_estimate(m, n, k, *t, 1, False))


@functools.lru_cache(maxsize=4096)
def mid_profitable(m: int, n: int, k: int, reduced: bool = True) -> bool:
    """Where this kernel beats the library GEMM on MI355X (padded weight rows, in graphs).  Where the next kernel sums the
    K-split slabs (not ``reduced``): one row through an 8B qkv projection 11.2 against 16.2 us, 2048 x 2048 5.5 / 8.5, but
    not once the slabs outweigh a small W (2048 x 2048 at 128 and 256 rows 9.9 / 8.9 and 13.3 / 10.2, 3072 x 3072 at 256
    16.5 / 17.7; 4608 x 3072 18.3 / 32).  With a reduction of its own (4 to 9 us): 48 rows into K >= 2 N, 128 into squarer
    shapes (from 48 when K >= 8192 and N <= 8192); small W stay with the library (3072 x 2048 at 256 rows 21 / 11).
    Outputs wide enough to fill the chip unsplit: always (an LM head of 128256 x 4096 at 1 / 64 / 256 rows 164 / 200 / 252 us,
    the library 190 / 222 / 309).  Above 256 rows W is read once a row tile: only where the library's tiles leave the chip idle as well,
    which they do for long reductions (8192 x 28672 at 384 and 512 rows 165 and 199 us / 201 and 313; 4096 x 14336 59 and 67 / 80
    and 91), and above 512 for fewer than 96 tiles of 256 x 256 (4096 x 14336 at 557, 768, 1024 and 1280 rows 74, 90, 113 and 133 /
    114, 107, 132 and 147; 3584 x 18944 at 768 102 / 183; 2048 x 8192 at 557 31 / 45; with 96 and more 8192 x 28672 at 557, 640 and
    900 rows 254, 287 and 357 / 258, 265 and 357, and squarer shapes at 557 32.8 / 36.9, 89 / 93, 101 / 97).  A reduction of its own leaves
    little of that above 768 rows where W is small and K hardly more than 2 N: 3584 x 7168 at 769, 1025 and 1150 rows 62, 74 and 75 / 55, 66
    and 71, with the next kernel's sums 61, 74 and 77 / 62, 74 and 79; 4096 x 8192 71, 85 and 87 / 76, 86 and 87."""
    if m <= 0 or m > MID_MAX_M or n < 512 or k < 1024:
        return False
    if m > 256:
        if reduced and m > 768 and 2 * k < 5 * n and n * k < 32 << 20:
            return False
        return k >= 2 * n and n * k >= 12 << 20 and (m <= 512 or -(-m // 256) * -(-n // 256) < 96)
    bm, bn, ksplit = mid_choose(m, n, k, reduced)
    if ksplit == 1:
        return _mid_blocks(m, n, bm, bn, 1) >= 192 and k >= 2048
    if not reduced:
        return n * k >= (2 << 20 if m <= 64 else 8 << 20 if m <= 128 else 12 << 20)
    if n > 12288 or k < 2048 or n * k < 12 << 20:
        return False
    return m >= 128 or (m >= 48 and (k >= 2 * n or (n <= 8192 and k >= 8192)))


MID_SILU_MIN_N, MID_SILU_MIN_K = 24576, 4096


def mid_silu_profitable(m: int, n: int, k: int) -> bool:
    """``[gate ; up]`` with the activation in the epilogue: outputs whose unsplit tiles fill the chip (14336 + 14336 columns:
    224 of 128).  8B at 1, 48 and 256 rows 41, 44 and 66 us (``stream_gemm`` 47, library and activation 75 and 82), 70B 152, 157
    and 190 (162, 166, 215).  Reductions below 4096 stay where they were: up to 8 rows ``stream_gemm``'s, above that the
    library's, though this kernel is ahead there too (37888 x 3584 at 16, 128 and 256 rows 61, 73 and 88 against 68, 85 and 93
    outside a graph; 28672 x 2048 22, 30 and 39 against 40, 39 and 48)."""
    return 0 < m <= 256 and n >= MID_SILU_MIN_N and k >= MID_SILU_MIN_K


def mid_gemm(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None, ksplit: Optional[int] = None,
             bm: Optional[int] = None, bn: Optional[int] = None, variant: Optional[int] = None,
             partials: bool = False, silu_mul: bool = False, bias: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``x [M<=1280, K] @ w [N, K]^T`` with W streamed once a tile of rows and K split over the chip.  ``partials``: the
    fp32 K-split slabs ``[ksplit, M, N]`` instead of their sum (None when the shape runs unsplit).  ``silu_mul``:
    ``w`` is ``[gate ; up]`` and ``silu(gate) * up`` (``N/2`` wide) the result.  ``bias [N]`` is added to the fp32 sums.  Calls written for
    the kernels before this one keep working: a tile wider than those in ``_MID_TILES`` runs as the widest of its rows, and
    ``variant``, which named one of two kernels that are one now, has no effect."""
    assert mid_supported(x, w, silu_mul), (x.shape, x.stride(), w.shape, w.stride(), x.dtype)
    assert not (silu_mul and (partials or (ksplit or 1) != 1))
    assert bias is None or (mid_bias_ok(bias, x, w) and not partials and not silu_mul)
    m, k = x.shape
    n = w.shape[0]
    if silu_mul:
        a, b = mid_silu_tile(m, n, k)
        c = 1
    else:
        a, b, c = mid_choose(m, n, k, not partials)
    bm = a if bm is None else bm
    bn = min(b if bn is None else bn, max(v for u, v in _MID_TILES if u == bm))
    ksplit = c if ksplit is None else ksplit
    assert 1 <= ksplit <= k // 64
    if partials:
        if ksplit <= 1:
            return None
        partial = torch.empty((ksplit, m, n), dtype=torch.float32, device=x.device)
        _check(_LIB.vdamd_mid_gemm(None, n, x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), None,
                                   partial.data_ptr(), m, n, k, ksplit, bm, bn, EPI_NONE, _dt(x), _stream()), "mid_gemm (partial sums)")
        return partial
    n_out = n // 2 if silu_mul else n
    if out is None:
        out = torch.empty((m, n_out), dtype=x.dtype, device=x.device)
    assert mid_out_ok(out, x, n_out)
    partial = torch.empty(ksplit * m * n, dtype=torch.float32, device=x.device) if ksplit > 1 else None
    _check(_LIB.vdamd_mid_gemm(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                               _ptr(bias), None if partial is None else partial.data_ptr(), m, n, k, ksplit, bm, bn,
                               EPI_SILU_MUL if silu_mul else EPI_NONE, _dt(x), _stream()), "mid_gemm")
    return out


# ------------------------------------- 256 x 256 tile LDS-DMA GEMM, M >= 512
BIG_MIN_M = 512
# with the SiLU*mul epilogue a single full row of tiles already beats library GEMM + activation kernel (70B gate_up at 256
# rows: 216 us against 229 + 9; profiles/r2_big_gemm_vs_library.txt); where mid_gemm takes the shape it is ahead of both (190)
BIG_MIN_M_SILU = 240
BIG_VARIANT = int(os.environ.get("VDAMD_BIG_GEMM_VARIANT", "0"))


def big_supported(x: torch.Tensor, w: torch.Tensor, silu_mul: bool = False) -> bool:
    return (x.dim() == 2 and w.dim() == 2 and x.shape[0] > 0 and x.dtype == w.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and x.shape[1] == w.shape[1]
            and w.shape[1] % 128 == 0 and w.shape[0] % (32 if silu_mul else 16) == 0
            and x.stride(1) == 1 and w.stride(1) == 1 and x.stride(0) % 8 == 0 and w.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and x.shape[0] * x.stride(0) * 2 < (1 << 32) - 64 and w.shape[0] * w.stride(0) * 2 < (1 << 32) - 64)


def big_profitable(m: int, n: int, k: int, silu_mul: bool = False) -> bool:
    """Where the 256 x 256-tile kernel is level with or ahead of the library GEMM on MI355X
    (benchmarks/big_gemm_bench.py, profiles/r2_big_gemm_vs_library.txt): enough tiles to fill the
    chip's 256 CUs in whole rounds.  With the SiLU*mul epilogue it also saves the activation kernel
    and wins at every batch size measured (512 .. 16384 rows); without it the library is 1-4 % ahead
    from 4096 rows up and stays in charge there."""
    if m < (BIG_MIN_M_SILU if silu_mul else BIG_MIN_M) or k < 1024:
        return False
    if m < BIG_MIN_M and m > 256:
        return False                  # between one and two full rows of tiles the second row is mostly padding
    tiles = -(-m // 256) * (-(-(n // 2) // 128) if silu_mul else -(-n // 256))
    rounds = -(-tiles // 256)
    eff = tiles / (rounds * 256.0)
    if silu_mul:
        return tiles >= 200 and eff >= 0.85
    return m <= 3072 and tiles >= 224 and eff >= 0.9


def big_gemm(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None,
             residual: Optional[torch.Tensor] = None, silu_mul: bool = False,
             variant: Optional[int] = None) -> torch.Tensor:
    """``x [M, K] @ w [N, K]^T`` on 256 x 256 tiles with both operands fed by LDS-DMA.  ``residual
    [M, N]`` is added in the epilogue; ``silu_mul`` treats ``w`` as ``[gate ; up]`` and returns
    ``silu(gate) * up`` (``N/2`` wide)."""
    assert big_supported(x, w, silu_mul), (x.shape, x.stride(), w.shape, w.stride(), x.dtype)
    assert not (silu_mul and residual is not None)
    m, k = x.shape
    n = w.shape[0]
    n_out = n // 2 if silu_mul else n
    if out is None:
        out = torch.empty((m, n_out), dtype=x.dtype, device=x.device)
    assert out.shape == (m, n_out) and out.dtype == x.dtype and out.stride(1) == 1 and out.data_ptr() % 16 == 0
    assert out.stride(0) % 8 == 0 and m * out.stride(0) * 2 < (1 << 32) - 64
    epi = EPI_SILU_MUL if silu_mul else (EPI_RESIDUAL if residual is not None else EPI_NONE)
    if residual is not None:
        assert (residual.shape == (m, n) and residual.dtype == x.dtype and residual.stride(1) == 1
                and residual.stride(0) % 4 == 0 and residual.data_ptr() % 8 == 0)
    _check(_LIB.vdamd_big_gemm(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                               None if residual is None else residual.data_ptr(),
                               0 if residual is None else residual.stride(0), m, n, k, epi,
                               BIG_VARIANT if variant is None else variant, _dt(x), _stream()), "big_gemm")
    return out


# ------------------------------------------------- grouped GEMMs (MoE experts)
def _check_tiles(tiles: torch.Tensor, x: torch.Tensor, tile_rows: int) -> int:
    assert tiles.dtype == torch.int32 and tiles.dim() == 2 and tiles.shape[1] == 3 and tiles.is_contiguous()
    assert tiles.device == x.device and tile_rows % 16 == 0
    assert x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
    return tiles.shape[0]


GROUPED_BIG_ROWS = 256             # rows per tile of the grouped form of the large-batch GEMM


def grouped_big_supported(x: torch.Tensor, w: torch.Tensor, silu_mul: bool = False) -> bool:
    """Whether the large-batch kernel's grouped form takes rows like ``x`` and experts ``w [G, N, K]``."""
    n, k = w.shape[1:]
    return (w.is_contiguous() and w.dtype in (torch.bfloat16, torch.float16) and w.dtype == x.dtype and k % 128 == 0
            and n % (32 if silu_mul else 16) == 0 and w.data_ptr() % 16 == 0 and n * k * 2 < (1 << 32) - 64)


def grouped_silu_supported(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the grouped GEMMs form ``silu(gate) * up`` of ``w = [gate ; up]`` themselves: halves of whole 16 columns, an expert's
    matrix within 32-bit byte offsets."""
    return w.shape[1] % 32 == 0 and w.shape[1] * w.shape[2] * 2 < (1 << 32) - 64


def grouped_gather_ok(x: torch.Tensor, src_row: torch.Tensor) -> bool:
    """Whether the grouped GEMMs can read the rows ``x[src_row]`` where they are: whole, aligned rows of x within 32-bit byte
    offsets, and eight entries at least (the large-batch kernel fetches that many at a time)."""
    return (x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.stride(0) >= x.shape[1] and x.data_ptr() % 16 == 0
            and x.shape[0] * x.stride(0) * 2 < (1 << 32) - 64 and src_row.numel() >= 8)


def grouped_gemm(x: torch.Tensor, w: torch.Tensor, tiles: torch.Tensor, tile_rows: int, out: Optional[torch.Tensor] = None,
                 silu_mul: bool = False, src_row: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[r] = x[r] @ w[g(r)]^T`` for group-sorted rows: ``w [G, N, K]``,
    ``tiles [n, 3] int32`` = (group, first row, rows <= tile_rows; 0 = unused).
    Every row covered by a tile must lie inside ``x``; rows outside all tiles
    are left untouched in ``out``.  ``tile_rows`` 256: the large-batch kernel, otherwise the short-batch one in tiles of 64 or 128
    rows.  ``silu_mul``: ``w = [gate ; up]`` and ``silu(gate) * up`` the result (``N / 2`` wide);
    ``src_row`` (with ``silu_mul``, at least eight): the tiles' rows are ``x[src_row]``, read where they are."""
    nt = _check_tiles(tiles, x, tile_rows)
    g, n, k = w.shape
    assert w.is_contiguous() and w.dtype == x.dtype and x.shape[1] == k
    assert k % 128 == 0 and n % (32 if silu_mul else 16) == 0 and (16 <= tile_rows <= 128 or tile_rows == GROUPED_BIG_ROWS)
    n_out = n // 2 if silu_mul else n
    rows = x.shape[0] if src_row is None else src_row.numel()
    if out is None:
        out = torch.empty((rows, n_out), dtype=x.dtype, device=x.device)
    assert src_row is None or (silu_mul and src_row.dtype == torch.int32 and src_row.is_contiguous() and src_row.is_cuda
                               and grouped_gather_ok(x, src_row))
    src = None if src_row is None else src_row.data_ptr()
    epi = EPI_SILU_MUL if silu_mul else EPI_NONE
    if tile_rows == GROUPED_BIG_ROWS:
        assert grouped_big_supported(x, w, silu_mul) and out.shape == (rows, n_out) and out.stride(1) == 1
        _check(_LIB.vdamd_big_gemm_grouped(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), k, n * k,
                                           tiles.data_ptr(), nt, src, x.shape[0], rows, n, k, epi, _dt(x), _stream()),
               "big_gemm_grouped")
        return out
    assert out.shape == (rows, n_out) and out.stride(1) == 1 and out.stride(0) % 4 == 0 and out.data_ptr() % 8 == 0
    if w.data_ptr() % 16:                  # (experts at an odd place of a larger buffer: their rows are fetched 16 bytes at a time)
        w = w.clone()
    _check(_LIB.vdamd_mid_gemm_grouped(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), k, n * k,
                                       tiles.data_ptr(), nt, src, x.shape[0], rows, n, k, 64 if tile_rows <= 64 else 128, 128, epi, _dt(x),
                                       _stream()),
           "mid_gemm_grouped")
    return out


W4_GROUPED_SILU_MAX_ROWS = 32      # tile sizes whose kernel forms silu(gate) * up while loading its operand


def grouped_w4a16_gemm(x: torch.Tensor, qw: torch.Tensor, sz: torch.Tensor, tiles: torch.Tensor,
                       tile_rows: int, out: Optional[torch.Tensor] = None, silu_mul: bool = False) -> torch.Tensor:
    """Grouped form of ``w4a16_gemm``: ``qw [G, N/16, K/128, 64, 4]``, ``sz [G, N/16, K/g, 16, 2]``.
    ``silu_mul`` (``tile_rows <= 32``): ``x`` is ``[rows, 2K] = [gate | up]`` and the left operand is
    ``silu(gate) * up``, formed inside the kernel."""
    nt = _check_tiles(tiles, x, tile_rows)
    assert qw.dim() == 5 and sz.dim() == 5 and qw.shape[0] == sz.shape[0] and tile_rows <= 64
    n, k, grp = _w4_dims(qw[0], sz[0])
    up_off = 0
    if silu_mul:
        assert tile_rows <= W4_GROUPED_SILU_MAX_ROWS and x.shape[1] == 2 * k
        up_off = k
    else:
        assert x.shape[1] == k
    assert qw.is_contiguous() and sz.is_contiguous() and x.dtype == sz.dtype
    if out is None:
        out = torch.empty((x.shape[0], n), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_w4a16_gemm_grouped(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), qw.data_ptr(),
                                         sz.data_ptr(), qw[0].numel(), sz[0].numel(), tiles.data_ptr(), nt,
                                         tile_rows, n, k, grp, _dt(x), up_off, _stream()), "w4a16_gemm_grouped")
    return out


def grouped_fp4a16_gemm(x: torch.Tensor, qw: torch.Tensor, fs: torch.Tensor, alpha: Optional[torch.Tensor],
                        tiles: torch.Tensor, tile_rows: int, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Grouped form of ``fp4a16_gemm``: ``qw [G, N/16, K/128, 64, 4]``, ``fs [G, N/16, K/128, 64]``,
    ``alpha [G, N]`` or None."""
    nt = _check_tiles(tiles, x, tile_rows)
    assert qw.dim() == 5 and fs.dim() == 4 and qw.shape[0] == fs.shape[0] and tile_rows <= 64
    n, k = _fp4_dims(qw[0], fs[0], None)
    assert qw.is_contiguous() and fs.is_contiguous() and x.shape[1] == k and _half(x)
    if alpha is not None:
        assert alpha.shape == (qw.shape[0], n) and alpha.dtype == torch.float32 and alpha.is_contiguous()
    if out is None:
        out = torch.empty((x.shape[0], n), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_fp4a16_gemm_grouped(out.data_ptr(), out.stride(0), x.data_ptr(), x.stride(0), qw.data_ptr(),
                                          fs.data_ptr(), qw[0].numel(), fs[0].numel() * 2,
                                          None if alpha is None else alpha.data_ptr(), tiles.data_ptr(), nt,
                                          tile_rows, n, k, _dt(x), _stream()), "fp4a16_gemm_grouped")
    return out


# ------------------------------------------------------------- MoE routing
MOE_MAX_EXPERTS = 512
MOE_MAX_TOPK = 16


def moe_topk(logits: torch.Tensor, k: int, renormalize: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    """softmax + top-k over router logits ``[T, E]``: ``(weights [T, k] fp32, experts [T, k] int32)``;
    ties go to the lowest expert id."""
    assert logits.dim() == 2 and logits.stride(1) == 1 and logits.dtype in _DT
    t, e = logits.shape
    assert k <= e <= MOE_MAX_EXPERTS and 1 <= k <= MOE_MAX_TOPK
    topw = torch.empty((t, k), dtype=torch.float32, device=logits.device)
    topi = torch.empty((t, k), dtype=torch.int32, device=logits.device)
    _check(_LIB.vdamd_moe_topk(logits.data_ptr(), logits.stride(0), topw.data_ptr(), topi.data_ptr(), t, e, k,
                               int(renormalize), _dt(logits), _stream()), "moe_topk")
    return topw, topi


def moe_topk_grouped(logits: torch.Tensor, bias: Optional[torch.Tensor], k: int, n_group: int, topk_group: int,
                     sigmoid: bool, group_top2: bool, renormalize: bool, scale: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """DeepSeek routing in one launch: scores = sigmoid (V3) or softmax (V2) of ``logits [T, E]``; experts chosen
    by ``score + bias`` inside the ``topk_group`` best of ``n_group`` groups (a group scored by its two best
    choices' sum, or by its best); weights = the chosen experts' unbiased scores, renormalised on request, times
    ``scale``.  Returns ``(weights [T, k] fp32, experts [T, k] int32)``."""
    assert logits.dim() == 2 and logits.stride(1) == 1 and logits.dtype in _DT
    t, e = logits.shape
    assert k <= e <= MOE_MAX_EXPERTS and 1 <= k <= MOE_MAX_TOPK and 1 <= n_group <= 64 and e % n_group == 0
    assert bias is None or (bias.dtype == torch.float32 and bias.numel() == e and bias.is_contiguous())
    topw = torch.empty((t, k), dtype=torch.float32, device=logits.device)
    topi = torch.empty((t, k), dtype=torch.int32, device=logits.device)
    _check(_LIB.vdamd_moe_topk_grouped(logits.data_ptr(), logits.stride(0), None if bias is None else bias.data_ptr(),
                                       topw.data_ptr(), topi.data_ptr(), t, e, k, n_group, max(1, topk_group),
                                       int(sigmoid), int(group_top2), int(renormalize), float(scale), _dt(logits),
                                       _stream()), "moe_topk_grouped")
    return topw, topi


def moe_align(topi: torch.Tensor, num_experts: int, tile_rows: int, expert_start: int = 0, local_experts: int = -1,
              ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Sort the ``T*k`` slots by expert on the device: ``(src_row [T*k] = token of each sorted row,
    inv [T*k] = sorted position of each slot, tiles [T*k // tile_rows + E, 3] int32)``.  Tiles of
    experts outside ``[expert_start, expert_start + local_experts)`` have 0 rows."""
    assert topi.dtype == torch.int32 and topi.dim() == 2 and topi.is_contiguous() and num_experts <= 1024
    t, k = topi.shape
    slots = t * k
    n = slots // tile_rows + num_experts
    src_row = torch.empty(slots, dtype=torch.int32, device=topi.device)
    inv = torch.empty(slots, dtype=torch.int32, device=topi.device)
    tiles = torch.empty((n, 3), dtype=torch.int32, device=topi.device)
    _check(_LIB.vdamd_moe_align(topi.data_ptr(), slots, k, num_experts, tile_rows, expert_start, local_experts,
                                src_row.data_ptr(), inv.data_ptr(), tiles.data_ptr(), n, _stream()), "moe_align")
    return src_row, inv, tiles


MOE_SMALL_MAX_TOKENS = 16


def moe_route_small(logits: torch.Tensor, x: torch.Tensor, k: int, renormalize: bool, tile_rows: int,
                    expert_start: int = 0, local_experts: int = -1):
    """``moe_topk`` + ``moe_align`` + the gather ``x[src_row]`` in one launch, for at most 16 tokens:
    ``(topw, topi, inv, tiles, xs [T*k, H])``.  Rows of one expert keep slot order."""
    nsplit, sstride = 1, 0
    if logits.dim() == 3:                       # fp32 partial sums of a K-split router GEMM, [splits, T, E]
        assert logits.dtype == torch.float32 and logits.is_contiguous()
        nsplit, sstride = logits.shape[0], logits.stride(0)
        logits = logits[0]
    t, e = logits.shape
    h = x.shape[1]
    assert logits.stride(1) == 1 and x.shape[0] == t and _half(x) and x.stride(1) == 1 and h % 8 == 0
    assert x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
    assert 1 <= t <= MOE_SMALL_MAX_TOKENS and k <= e <= MOE_MAX_EXPERTS and 1 <= k <= MOE_MAX_TOPK
    assert logits.dtype in (x.dtype, torch.float32)
    slots = t * k
    n = slots // tile_rows + e
    dev = x.device
    topw = torch.empty((t, k), dtype=torch.float32, device=dev)
    ints = torch.empty(3 * slots + 3 * n, dtype=torch.int32, device=dev)          # one allocation for the tables
    topi, src_row, inv = ints[:slots].view(t, k), ints[slots:2 * slots], ints[2 * slots:3 * slots]
    tiles = ints[3 * slots:].view(n, 3)
    xs = torch.empty((slots, h), dtype=x.dtype, device=dev)
    _check(_LIB.vdamd_moe_route_small(logits.data_ptr(), logits.stride(0), t, e, k, int(renormalize), tile_rows,
                                      expert_start, local_experts, topw.data_ptr(), topi.data_ptr(),
                                      src_row.data_ptr(), inv.data_ptr(), tiles.data_ptr(), n, x.data_ptr(),
                                      x.stride(0), xs.data_ptr(), h, _dt(logits), _dt(x), nsplit, sstride, _stream()),
           "moe_route_small")
    return topw, topi, inv, tiles, xs


def moe_combine(y: torch.Tensor, topw: Optional[torch.Tensor], topi: torch.Tensor, inv: torch.Tensor, expert_start: int = 0,
                local_experts: int = -1, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[t] = sum_j topw[t, j] * y[inv[t*k + j]]`` in fp32 (``topw`` None: weights of one; slots of experts this rank does not hold are skipped).
    ``bias [local experts, H]``: each row first gains its expert's bias (rounded to the row's dtype)."""
    t, k = topi.shape
    h = y.shape[1]
    if bias is not None:
        assert bias.dtype == y.dtype and bias.dim() == 2 and bias.shape[1] == h and bias.is_contiguous()
        assert bias.shape[0] >= (local_experts if local_experts >= 0 else 1)
    assert _half(y) and y.stride(1) == 1 and y.stride(0) % 8 == 0 and h % 8 == 0 and y.data_ptr() % 16 == 0
    assert topw is None or (topw.dtype == torch.float32 and topw.is_contiguous())
    assert topi.is_contiguous() and inv.numel() == t * k
    out = torch.empty((t, h), dtype=y.dtype, device=y.device)
    _check(_LIB.vdamd_moe_combine(out.data_ptr(), h, y.data_ptr(), y.stride(0), _ptr(topw), topi.data_ptr(),
                                  inv.data_ptr(), t, k, h, expert_start, local_experts,
                                  None if bias is None else bias.data_ptr(), _dt(y), _stream()),
           "moe_combine")
    return out


def bias_clamped_glu(h: torch.Tensor, bias: torch.Tensor, topi: torch.Tensor, inv: torch.Tensor, expert_start: int,
                     local_experts: int, limit: float, alpha: float) -> torch.Tensor:
    """gpt-oss expert activation on expert-sorted rows ``h [rows, 2 ip] = [gate | up]``: every row gains the
    ``[2 ip]`` bias of its expert, then ``(up + 1) * gate * sigmoid(alpha * gate)`` with ``gate`` clamped from
    above and ``up`` on both sides; returns ``[rows, ip]``.  Rows of slots whose expert lives elsewhere are
    left unwritten (their weights are zero in the combine)."""
    rows, two_ip = h.shape
    ip = two_ip // 2
    slots = topi.numel()
    assert _half(h) and h.stride(1) == 1 and ip % 8 == 0 and inv.numel() == slots and rows >= slots
    assert bias.dtype == h.dtype and bias.shape[1] == two_ip and bias.is_contiguous()
    assert topi.dtype == torch.int32 and inv.dtype == torch.int32 and topi.is_contiguous() and inv.is_contiguous()
    out = torch.empty((rows, ip), dtype=h.dtype, device=h.device)
    _check(_LIB.vdamd_bias_clamped_glu(out.data_ptr(), ip, h.data_ptr(), h.stride(0), bias.data_ptr(), topi.data_ptr(),
                                       inv.data_ptr(), slots, ip, expert_start, local_experts, float(limit),
                                       float(alpha), _dt(h), _stream()), "bias_clamped_glu")
    return out


def moe_combine_add_rms_norm(y: torch.Tensor, topw: torch.Tensor, topi: torch.Tensor, inv: torch.Tensor,
                             expert_start: int, local_experts: int, residual: torch.Tensor, weight: torch.Tensor,
                             eps: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """``moe_combine`` followed by ``fused_add_rms_norm`` in one launch: ``residual`` (in place) gains the
    weighted sum of each token's expert rows, and its RMSNorm is returned next to it."""
    t, k = topi.shape
    h = y.shape[1]
    assert y.stride(1) == 1 and h % 8 == 0 and h <= 32768 and k <= 16 and _half(y)
    assert residual.shape == (t, h) and residual.is_contiguous() and residual.dtype == y.dtype == weight.dtype
    assert topw.dtype == torch.float32 and topw.is_contiguous() and topi.is_contiguous() and inv.is_contiguous()
    out = torch.empty_like(residual)
    _check(_LIB.vdamd_moe_combine_add_rms_norm(out.data_ptr(), h, y.data_ptr(), y.stride(0), topw.data_ptr(),
                                               topi.data_ptr(), inv.data_ptr(), t, k, h, expert_start, local_experts,
                                               residual.data_ptr(), weight.data_ptr(), float(eps), _dt(y), _stream()),
           "moe_combine_add_rms_norm")
    return out, residual


# ------------------------------------------------------------------ FP8 W8A8
def dynamic_fp8_quant(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-token dynamic quantisation to OCP e4m3: ``(xq [M, K] float8_e4m3fn, scale [M, 1] fp32)``
    with ``x ~ xq * scale``."""
    assert x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
    m, k = x.shape
    out = torch.empty((m, k), dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty((m, 1), dtype=torch.float32, device=x.device)
    _check(_LIB.vdamd_dynamic_fp8_quant(out.data_ptr(), scale.data_ptr(), x.data_ptr(), m, k, x.stride(0),
                                        _dt(x), _stream()), "dynamic_fp8_quant")
    return out, scale


# ------------------------------------------------ multi-head latent attention (DeepSeek) over a latent cache
MLA_KERNEL_DIMS = ((576, 512), (320, 256), (96, 64))


def mla_supported(dk: int, dv: int, dtype: torch.dtype) -> bool:
    return (dk, dv) in MLA_KERNEL_DIMS and dtype in (torch.bfloat16, torch.float16)


def _mla_fp8(k_cache: torch.Tensor, v_cache: torch.Tensor, dtype: torch.dtype) -> int:
    """1 when the latent caches hold e4m3 bytes, 0 when elements of the model type."""
    assert k_cache.dtype == v_cache.dtype and k_cache.dtype in (dtype, torch.float8_e4m3fn), (k_cache.dtype, dtype)
    return int(k_cache.dtype == torch.float8_e4m3fn)


def mla_cache_write(latent: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                    slot_mapping: torch.Tensor) -> None:
    """``latent[T, DK]`` (normalised c_kv | rotated k_rope) into the key-row cache and, its first DV values,
    into the V^T fragment cache."""
    t, dk = latent.shape
    dv = v_cache.shape[2] * v_cache.shape[4]
    bs = k_cache.shape[2]
    assert latent.stride(1) == 1 and k_cache.shape[1] == 1 and k_cache.shape[3] == dk and k_cache.is_contiguous()
    fp8 = _mla_fp8(k_cache, v_cache, latent.dtype)
    assert v_cache.is_contiguous() and v_cache.shape[3] * v_cache.shape[5] == bs
    assert slot_mapping.dtype == torch.int32 and slot_mapping.numel() >= t
    _check(_LIB.vdamd_mla_cache_write(latent.data_ptr(), latent.stride(0), k_cache.data_ptr(), v_cache.data_ptr(),
                                      slot_mapping.data_ptr(), t, dk, dv, bs, _dt(latent), fp8, _stream()),
           "mla_cache_write")


def mla_rows_ok(k_cache: torch.Tensor, dv: int) -> bool:
    """Whether the kernel that takes the values from the key rows reads this cache (16-bit rows, whole groups of 32 keys in a
    block, a value width that divides over its waves)."""
    return k_cache.dtype != FP8_KV and k_cache.shape[2] % 32 == 0 and dv % 256 == 0


def mla_num_splits(tokens: int, q_tiles: int, max_seq_len: int, workgroups: int = 256) -> int:
    """KV splits of the kernel that reads both caches: about one workgroup per CU in total and no split shorter than two groups
    of 32 keys.  A workgroup streams ~36 GB/s by itself (one group in flight ahead of the one being multiplied), so the chip's
    bandwidth needs a few hundred of them; beyond that, more splits only add partial sums to write and merge
    (scripts/dev/mla_split_sweep.py).  A merge costs ~2 us: 16 heads over 500 keys take 21 us in 2 splits, 12.5 in 7."""
    want = -(-workgroups // max(1, tokens * q_tiles))
    return int(max(1, min(want, max_seq_len // 64, 64)))


def mla_plan(tokens: int, heads: int, keys: int, by_token: bool, seqs: int, rows_ok: bool, mode: Optional[int] = None,
             captured: bool = True) -> Tuple[int, int]:
    """Kernel (``mla_attention``'s ``mode``, chosen here when None) and KV splits of a step of ``tokens`` rows of up to ``keys`` keys
    from ``seqs`` sequences (``by_token``: rows name theirs), ``captured`` in a graph or launched from Python.

    The kernel over the key rows (3) wherever it reads the cache (``rows_ok``): it reads a row once per token and 16 heads, but out of
    the caches and by DMA; the two that share keys between four tiles (1, 2) read both caches into registers, 70 KB per 5 us a
    workgroup.  us, shared / rows: prompt tokens of 16 heads, 2611 of three sequences 377 / 232, 1834 of one 419 / 236, 85 behind 330
    34 / 21, four each of 64 sequences of 4000 keys 664 / 182, of 16 of 1000 58 / 24; of 128 heads, 880 of three 902 / 584, 76 77 / 31,
    565 of 5000 keys 3647 / 2255; decoded rows of 128 heads, 69 of 780 keys 167 / 101, 20 of 3000 124 / 101, 128 of 600 139 / 112; of
    64, 100 of 800 104 / 68, 256 of 1500 346 / 288.

    Splits make as many workgroups as run at once - one per CU of the kernels that share keys, two of the one over key rows - and not
    more: what is left over waits for a second round.  Over key rows 100 decoded rows of 700 keys 26.8 in 5 and 32.6 in 6, 160 of 3000
    keys 93 in 3 and 117 in 4.  Over both caches a prompt of 200 tokens, 16 heads, 700 keys (50 workgroups) 47 us in 5 splits, 66 in 6;
    three of 64, 32 heads, 564 keys (102) 65 in 2, 92 in 3; prompts that take most CUs whole still go in two, which evens out their
    rows of different lengths (two of 500 rows on average behind 500 keys: 269 us whole, 227 in 2; one of 700: 116 and 102; though two
    of exactly 300: 58 and 62).  Splits hold 64 keys, or 128 where more than 64 workgroups leave many partial sums (16 rows of 128
    heads, 200 keys: 14.5 us whole, 19.7 in 3), 256 where there is a workgroup for every CU (256 rows, 400 keys: 24.7 whole, 32.8
    in 2).
    Outside a graph a second launch and its buffers cost the host 6.5 us: up to 383 keys rows are not split (a decoded row of 200 keys
    13.6 us whole, 20 in 3; 32 prompt tokens of 300 keys 17.0 and 21.2, 8 of 380 19.7 and 21.0; 500 keys 25 and 20)."""
    q_tiles = -(-heads // 16)
    if mode is None:
        # (four head tiles per workgroup need enough workgroups left to fill the chip)
        mode = 3 if rows_ok else 1 if by_token else 2 if q_tiles >= 4 and tokens * q_tiles >= 128 else 0
    if mode in (0, 3, 4) and keys < 384 and not captured:
        return mode, 1
    if mode == 0:
        return mode, mla_num_splits(tokens, q_tiles, keys)
    if mode == 1:
        wgs = min(tokens, -(-tokens // 4) + seqs - 1) * q_tiles       # (a sequence's tokens start a group of four anywhere)
    else:
        wgs = tokens * (-(-q_tiles // 4) if mode in (2, 4) else q_tiles)
    per, shortest = (512 if mode == 3 else 256) // max(wgs, 1), 64
    if mode == 1 and 128 < wgs < 256:
        per = 2
    if mode == 3 and wgs > 64:
        shortest = 128 if wgs < 256 else 256
    if mode == 4:
        # (us of a call, 128 heads: 50 and 64 rows of 400 keys in one split 29 and 30, in two 44 and 49, single tiles 34 and 41; 32 rows of
        # 800 in two and four 43 and 48; 50 of 1500 in one and two 68 and 65; 20 of 600 in one and three 42 and 34)
        shortest = 192 if wgs <= 48 else 320
    return mode, max(1, min(per, keys // shortest, 64))


def mla_heads_shared(tokens: int, heads: int, keys: int, captured: bool, prompts: int = 0) -> bool:
    """Whether a step over key rows (``mla_plan``'s 3) goes four tiles of 16 heads a workgroup (4): from 64 heads on, where there is
    work enough.  Such a workgroup needs the time of two single ones for four tiles of a key, and 6 to 8 us more before its first
    product and after its last, so the line is at 160000 (tiles - what the last four leave idle) x rows x keys.  us, single / shared:
    128 heads, 50 rows of 250 keys 29 / 26, 100 of 250 46 / 29, 20 of 1500 62 / 43, 12 of 4000 86 / 49, 5 of 4000 39 / 36, 3 of 9000
    52 / 39; 64 heads, 12 of 4000 49 / 38, 50 of 1500 78 / 47, 100 of 1500 132 / 67; below the line, 128 heads, one row of 3000 20 / 26,
    8 of 1500 31 / 34, 20 of 600 34 / 36, and 64 heads, 8 of 4000 34 / 37, 20 of 600 25 / 32.
    In a graph ``keys`` is a bound that the lengths may be far below, and a split that is empty still costs its partial sums: only
    steps whose workgroups fill half of the CUs whole (100 rows of 128 heads, 100 keys: 27 / 22; of 20 keys and fewer 12 / 14, 512 rows
    42 / 57, which no bound tells).
    The rows of ``prompts`` sequences see fewer keys than the longest of them: half as many where nothing lies in front, and hardly
    any in short ones (200 tokens of 96 heads 28 / 33, four prompts of 100 of 128 heads 47 / 53).  80 heads, five tiles in eight
    places, gain less (300 tokens 44 / 48, and 28 / 34 of 320 values; 700 162 / 134; 130 behind 1000 of 320 values 67 / 70), and
    several prompts may be shorter than the longest tells (five of 30 to 512 153 / 159, 98 / 106)."""
    q_tiles = -(-heads // 16)
    fours = -(-q_tiles // 4)
    least = 160000
    if prompts > 0:
        new = tokens / prompts
        keys = keys - new / 2 if new <= keys else keys           # (more rows than keys: a window)
        if keys < 100:
            return False
        if q_tiles % 4 == 1:
            least = 300000 if prompts == 1 else 1000000
    if q_tiles < 4 or tokens * keys * (2 * q_tiles - 4 * fours) < least:
        return False
    return not captured or tokens * fours > 128


# latent rows of a decode step that are read past the caches (again and again 57 and 86 MB are slower so, 210 MB 63 -> 57 us)
LATENT_ONCE_BYTES = 128 << 20


def mla_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, block_table: torch.Tensor,
                  token_seq: Optional[torch.Tensor], seq_lens: torch.Tensor, scale: float, max_seq_len: int,
                  out: Optional[torch.Tensor] = None, splits: Optional[int] = None,
                  mode: Optional[int] = None, precise: bool = False, window: int = 0,
                  sinks: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``q[T, Hq, DK]`` against the latent cache -> ``[T, Hq, DV]``; token ``t`` reads block-table row
    ``token_seq[t]`` (``t`` itself when None) and sees keys ``0 .. seq_lens[t] - 1``.  ``mode`` (default: by
    shape): 0 = a workgroup per (token, 16 heads); 1 = four consecutive tokens of a sequence per workgroup
    (steps with ``token_seq``: prefill chunks, verification - the tokens of a sequence must be adjacent rows at
    consecutive positions); 2 = four head tiles of a token per workgroup (64 heads per rank and more); 3 = as 0,
    the values read from the key rows (their first ``DV`` values, which is what every writer puts into both caches):
    half the bytes, 1.1 to 4.6 times as fast from one sequence of 32 keys to 256 of 1500 and prompts of 5000, at every width and
    head count measured, so the others are left with what 3 does not read (``mla_rows_ok``); 4 = four head tiles of a token per
    workgroup over the key rows, the default where that is faster (``mla_heads_shared``; weights not ``precise``).
    ``precise``: the softmax weights enter the PV product with fp32 precision (a high and a low 16-bit part).
    ``window`` > 0: only the last ``window`` of those keys; ``sinks[Hq]`` (fp32): ``exp(sinks[h])`` joins head ``h``'s
    softmax denominator; ``gate[T, Hq]`` (raw, rows may be strided): the output times its sigmoid."""
    t, hq, dk = q.shape
    dv = v_cache.shape[2] * v_cache.shape[4]
    bs = k_cache.shape[2]
    assert mla_supported(dk, dv, q.dtype), (dk, dv, q.dtype)
    assert q.stride(2) == 1 and q.stride(1) == dk and k_cache.is_contiguous() and v_cache.is_contiguous()
    assert block_table.dtype == torch.int32 and block_table.stride(1) == 1 and seq_lens.dtype == torch.int32
    assert seq_lens.numel() >= t and (token_seq is None or (token_seq.dtype == torch.int32 and token_seq.numel() >= t))
    assert token_seq is not None or block_table.shape[0] >= t
    if out is None:
        out = torch.empty((t, hq, dv), dtype=q.dtype, device=q.device)
    assert out.stride(2) == 1 and out.stride(1) == dv
    gate_stride = 0
    if gate is not None:
        assert gate.dim() == 2 and gate.shape[0] >= t and gate.shape[1] == hq and gate.stride(1) == 1 and gate.dtype == q.dtype
        gate_stride = gate.stride(0)
    keys = min(max_seq_len, int(window) + 3) if window else max_seq_len
    asked = mode
    mode, best = mla_plan(t, hq, keys, token_seq is not None, block_table.shape[0], mla_rows_ok(k_cache, dv), mode,
                          keys >= 384 or keys >= 128 and torch.cuda.is_current_stream_capturing())
    if (asked is None and mode == 3 and not precise and hq > 48
            and mla_heads_shared(t, hq, keys, torch.cuda.is_current_stream_capturing(),
                                 block_table.shape[0] if token_seq is not None else 0)):
        mode, best = mla_plan(t, hq, keys, token_seq is not None, block_table.shape[0], True, 4, keys >= 384)
    # (a bound, in a graph a loose one: the kernel asks the lengths, and which pages several rows share)
    past = max(1, LATENT_ONCE_BYTES) if (mode == 3 and hq <= 16 and token_seq is None
                                         and t * keys * dk * 2 >= LATENT_ONCE_BYTES) else 0
    splits = best if splits is None else splits
    part_o = part_ml = None
    if splits > 1:
        part_o = torch.empty((t * hq * splits, dv), dtype=torch.float32, device=q.device)
        part_ml = torch.empty((t * hq * splits, 2), dtype=torch.float32, device=q.device)
    _check(_LIB.vdamd_mla_attention(
        out.data_ptr(), out.stride(0), None if part_o is None else part_o.data_ptr(),
        None if part_ml is None else part_ml.data_ptr(), q.data_ptr(), q.stride(0), k_cache.data_ptr(),
        v_cache.data_ptr(), block_table.data_ptr(), block_table.stride(0),
        None if token_seq is None else token_seq.data_ptr(), seq_lens.data_ptr(), float(scale), t, hq, dk, dv, bs,
        splits, int(mode), _dt(q), _mla_fp8(k_cache, v_cache, q.dtype), int(bool(precise)), int(window),
        _ptr(_f32_vec(sinks, hq, "sinks")), _ptr(gate), gate_stride, past, _stream()), "mla_attention")
    return out


def mla_prep(q: torch.Tensor, nope: int, q_lat: torch.Tensor, latent: torch.Tensor, norm_weight: torch.Tensor,
             eps: float, cos_sin: torch.Tensor, positions: torch.Tensor, k_cache: Optional[torch.Tensor],
             v_cache: Optional[torch.Tensor], slot_mapping: Optional[torch.Tensor]) -> torch.Tensor:
    """One launch between the projections and the attention of a latent-cache layer: the latent row of every
    token normalised (first ``rank`` values) and rotated (last ``rope`` values) into both cache forms, and the
    absorbed query ``[T, H, rank + rope] = [q_lat | rotated q[..., nope:]]`` returned.  ``q [T, H, nope + rope]``
    and ``q_lat [H, T, rank]`` may be strided views; without a cache (``slot_mapping`` None) only the query is made."""
    t, h, qd = q.shape
    rank = q_lat.shape[2]
    rope = qd - nope
    assert q.stride(2) == 1 and q_lat.stride(2) == 1 and latent.stride(1) == 1 and latent.shape == (t, rank + rope)
    assert q_lat.shape == (h, t, rank) and cos_sin.dtype == torch.float32 and cos_sin.shape[1] == rope
    assert positions.dtype == torch.int32 and norm_weight.dtype == q.dtype == q_lat.dtype == latent.dtype
    out = torch.empty((t, h, rank + rope), dtype=q.dtype, device=q.device)
    bs, fp8 = 8, 0
    if slot_mapping is not None:
        bs = k_cache.shape[2]
        assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[3] == rank + rope
        assert slot_mapping.dtype == torch.int32 and slot_mapping.numel() >= t
        fp8 = _mla_fp8(k_cache, v_cache, q.dtype)
    _check(_LIB.vdamd_mla_prep(out.data_ptr(), q.data_ptr(), q.stride(0), q.stride(1), nope, q_lat.data_ptr(),
                               q_lat.stride(0), q_lat.stride(1), latent.data_ptr(), latent.stride(0),
                               norm_weight.data_ptr(), float(eps), cos_sin.data_ptr(), positions.data_ptr(),
                               None if slot_mapping is None else k_cache.data_ptr(),
                               None if slot_mapping is None else v_cache.data_ptr(),
                               None if slot_mapping is None else slot_mapping.data_ptr(), t, h, rank, rope, bs,
                               _dt(q), fp8, _stream()), "mla_prep")
    return out


# ------------------------------------------------ single-gain norms, PolyNorm, convolved q/k/v, windowed attention
def _i32(t: Optional[torch.Tensor], name: str) -> Optional[torch.Tensor]:
    if t is None:
        return None
    assert t.dtype == torch.int32 and t.is_contiguous() and t.is_cuda, f"{name}: int32 contiguous device tensor expected"
    return t


def _f32_vec(t: Optional[torch.Tensor], n: int, name: str) -> Optional[torch.Tensor]:
    if t is None:
        return None
    assert t.dtype == torch.float32 and t.is_cuda and t.numel() == n and t.is_contiguous(), \
        f"{name}: {n} contiguous fp32 values expected, got {tuple(t.shape)} {t.dtype}"
    return t


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def embed_positions(ids: torch.Tensor, positions: torch.Tensor, embed: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    t, h = ids.shape[0], embed.shape[1]
    assert ids.dim() == 1 and positions.shape[0] >= t and embed.is_contiguous() and pos.is_contiguous()
    assert pos.shape[1] == h and pos.dtype == embed.dtype
    ids = ids if ids.dtype == torch.int32 else ids.to(torch.int32)
    positions = positions if positions.dtype == torch.int32 else positions.to(torch.int32)
    out = torch.empty((t, h), dtype=torch.float32, device=embed.device)
    _check(_LIB.vdamd_embed_positions(out.data_ptr(), _i32(ids, "ids").data_ptr(), _i32(positions, "positions").data_ptr(),
                                      embed.data_ptr(), pos.data_ptr(), t, h, embed.shape[0], pos.shape[0], _dt(embed),
                                      _stream()), "embed_positions")
    return out


def scalar_rms_norm(x: torch.Tensor, gain: torch.Tensor, eps: float, out_dtype: torch.dtype) -> torch.Tensor:
    h = x.shape[-1]
    x2 = x.reshape(-1, h)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    out = torch.empty((x2.shape[0], h), dtype=out_dtype, device=x.device)
    _check(_LIB.vdamd_scalar_norm(out.data_ptr(), x2.data_ptr(), _f32_vec(gain, 1, "gain").data_ptr(), float(eps),
                                  x2.shape[0], h, x2.stride(0), _dt(x2), _dt(out), _stream()), "scalar_norm")
    return out.view(x.shape[:-1] + (h,))


def scalar_norm_residual(y: torch.Tensor, post_gain: torch.Tensor, residual: torch.Tensor,
                         next_gain: Optional[torch.Tensor], eps: float, out_dtype: torch.dtype):
    t, h = y.shape
    assert residual.shape == (t, h) and residual.dtype == torch.float32 and residual.is_contiguous() and y.stride(1) == 1
    out = torch.empty((t, h), dtype=out_dtype, device=y.device) if next_gain is not None else None
    _check(_LIB.vdamd_scalar_norm_residual(
        _ptr(out), y.data_ptr(), residual.data_ptr(), _f32_vec(post_gain, 1, "post_gain").data_ptr(),
        _ptr(_f32_vec(next_gain, 1, "next_gain")), float(eps), t, h, y.stride(0), _dt(y),
        _DT[out_dtype], _stream()), "scalar_norm_residual")
    return out


def poly_norm(z: torch.Tensor, coef: torch.Tensor, eps: float) -> torch.Tensor:
    f = z.shape[-1]
    z2 = z.reshape(-1, f)
    if z2.stride(-1) != 1:
        z2 = z2.contiguous()
    out = torch.empty((z2.shape[0], f), dtype=z.dtype, device=z.device)
    _check(_LIB.vdamd_poly_norm(out.data_ptr(), z2.data_ptr(), _f32_vec(coef, 4, "coef").data_ptr(), float(eps),
                                z2.shape[0], f, z2.stride(0), _dt(z2), _stream()), "poly_norm")
    return out.view(z.shape)


CONV_MAX_TAPS = 16
UNIT_MAX_WIDTH = 512
# the matrix-core attention kernel where the shape allows it (tests switch it off to run the plain kernel in bf16)
WINDOW_ATTENTION_MFMA = os.environ.get("VDAMD_WINDOW_ATTENTION_MFMA", "1") != "0"
CROSS_GROUP_PROMPT = int(os.environ.get("VDAMD_CROSS_GROUP_PROMPT", "4"))
CROSS_GROUP_DECODE = int(os.environ.get("VDAMD_CROSS_GROUP_DECODE", "2"))


def conv_norm_cache(x, conv_weight, state, slots, query_start_loc, seq_lens, token_seq, positions, num_heads: int,
                    num_kv_heads: int, dim: int, vdim: int, q_norm, k_norm, eps: float, v_first, v_lambda,
                    keep_v: bool, k_cache, v_cache, slot_mapping, has_prefill: bool = True, inv_freq=None):
    t = x.shape[0]
    c = num_heads * dim + num_kv_heads * (dim + vdim)
    taps = conv_weight.shape[0]
    r = max(taps - 1, 1)
    b = seq_lens.shape[0]
    assert x.dim() == 2 and x.shape[1] >= c and x.stride(1) == 1 and x.is_cuda
    assert conv_weight.shape == (taps, c) and conv_weight.dtype == x.dtype and conv_weight.is_contiguous()
    assert 1 <= taps <= CONV_MAX_TAPS and dim <= UNIT_MAX_WIDTH and vdim <= UNIT_MAX_WIDTH
    assert state is not None and state.dtype == x.dtype and state.is_contiguous() and state.shape[1:] == (r, c), \
        (None if state is None else state.shape, (r, c))
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1 and positions.shape[0] >= t
    assert slot_mapping.shape[0] >= t and (token_seq is None or token_seq.shape[0] >= t)
    assert token_seq is not None or t <= b, "rows without a sequence"
    if slots.dtype != torch.int32:
        slots = slots.to(torch.int32)
    if k_cache is not None:
        bs = k_cache.shape[2]
        assert k_cache.dtype == x.dtype and v_cache.dtype == x.dtype and k_cache.is_contiguous() and v_cache.is_contiguous()
        assert k_cache.shape[1:] == (num_kv_heads, bs, dim) and bs % 8 == 0
        assert v_cache.shape == (k_cache.shape[0], num_kv_heads, bs // 8, vdim, 8)
    else:
        bs = 1
    gv = num_kv_heads * vdim
    if v_first is not None:
        assert v_first.shape == (t, gv) and v_first.dtype == torch.float32 and v_first.is_contiguous()
    q = torch.empty((t, num_heads, dim), dtype=x.dtype, device=x.device)
    kept = torch.empty((t, gv), dtype=torch.float32, device=x.device) if keep_v else None
    half = 0 if inv_freq is None else int(inv_freq.numel())
    assert 2 * half <= dim and (q_norm is None) == (k_norm is None)
    _check(_LIB.vdamd_conv_norm_cache(
        x.data_ptr(), x.stride(0), conv_weight.data_ptr(), state.data_ptr(), _i32(slots, "slots").data_ptr(),
        _i32(query_start_loc, "query_start_loc").data_ptr(), _i32(seq_lens, "seq_lens").data_ptr(),
        _ptr(_i32(token_seq, "token_seq")), _i32(positions, "positions").data_ptr(),
        _ptr(_f32_vec(q_norm, dim, "q_norm")), _ptr(_f32_vec(k_norm, dim, "k_norm")),
        _ptr(v_first), _ptr(_f32_vec(v_lambda, 1, "v_lambda")) if v_first is not None else None, _ptr(kept),
        q.data_ptr(), _ptr(k_cache), _ptr(v_cache), _i32(slot_mapping, "slot_mapping").data_ptr(),
        t, b, num_heads, num_kv_heads, dim, vdim, taps, bs, float(eps), 1 if has_prefill else 0,
        _ptr(_f32_vec(inv_freq, half, "inv_freq")) if half else None, half, _dt(x), _stream()),
        "conv_norm_cache")
    return q, kept


def window_bias_attention(q, k_cache, v_cache, block_table, query_start_loc, seq_lens, token_seq, positions,
                          scale: float, softcap: float, window: int, keep_first: int, bias_scale, bias_rate, sinks,
                          gate, max_query_len: int = 0, out=None, chunk: int = 0, crossed: bool = False):
    """``crossed``: every query head's weights on every value head, fp32 ``[T, H, Hkv, Dv]``."""
    t, h, d = q.shape
    g, bs, dv = k_cache.shape[1], k_cache.shape[2], v_cache.shape[3]
    b = seq_lens.shape[0]
    assert q.is_contiguous() and q.dtype == k_cache.dtype == v_cache.dtype and h % g == 0
    assert k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[3] == d
    assert v_cache.shape == (k_cache.shape[0], g, bs // 8, dv, 8) and bs % 8 == 0 and dv <= UNIT_MAX_WIDTH
    assert query_start_loc.shape[0] >= b + 1 and block_table.shape[0] >= b
    assert block_table.dim() == 2 and block_table.stride(1) == 1 and block_table.dtype == torch.int32
    assert positions.shape[0] >= t and (token_seq is None or token_seq.shape[0] >= t)
    assert token_seq is not None or t <= block_table.shape[0], "rows without a sequence"
    gate_stride = 0
    if gate is not None:
        assert gate.shape == (t, h) and gate.stride(1) == 1 and gate.dtype == q.dtype
        gate_stride = gate.stride(0)
    out_shape, out_dtype = ((t, h, g, dv), torch.float32) if crossed else ((t, h, dv), q.dtype)
    # value heads that share one computation of the scores: four where the rows fill the matrix cores (prompt
    # portions); decoded rows are bound by the loads in flight, and two leave more waves resident (measured)
    cross = 0 if not crossed else (CROSS_GROUP_DECODE if max_query_len == 1 else CROSS_GROUP_PROMPT)
    assert not crossed or (gate is None and sinks is None)
    if out is None:
        out = torch.empty(out_shape, dtype=out_dtype, device=q.device)
    assert out.shape == out_shape and out.dtype == out_dtype and out.is_contiguous()
    _check(_LIB.vdamd_window_bias_attention(
        q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr(), block_table.stride(0),
        _ptr(_i32(token_seq, "token_seq")), _i32(positions, "positions").data_ptr(),
        _i32(query_start_loc, "query_start_loc").data_ptr(), _i32(seq_lens, "seq_lens").data_ptr(),
        _ptr(_f32_vec(bias_scale, h, "bias_scale")), _ptr(_f32_vec(bias_rate, h, "bias_rate")),
        _ptr(_f32_vec(sinks, h, "sinks")), _ptr(gate), gate_stride, out.data_ptr(), t, b, h, g, d, dv, bs,
        int(window), int(keep_first), int(max_query_len) if max_query_len else t, float(scale), float(softcap),
        1 if WINDOW_ATTENTION_MFMA else 0, int(chunk), cross, _dt(q), _stream()), "window_bias_attention")
    return out


# ------------------------------------------------ fp32 residual stream with layer norms, decayed linear attention,
# ------------------------------------------------ gated norm, clamped GLU, latent attention over one row cache
def embed_scaled(ids: torch.Tensor, weight: torch.Tensor, scale: float) -> torch.Tensor:
    t, h = ids.numel(), weight.shape[1]
    assert ids.dtype == torch.int32 and weight.is_contiguous()
    out = torch.empty((t, h), dtype=torch.float32, device=weight.device)
    _check(_LIB.vdamd_embed_scaled(out.data_ptr(), ids.data_ptr(), weight.data_ptr(), float(scale), t, h,
                                   weight.shape[0], _dt(weight), _stream()), "embed_scaled")
    return out


def layer_norm_to(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float,
                  out_dtype: torch.dtype) -> torch.Tensor:
    t, h = x.shape
    assert x.stride(1) == 1
    out = torch.empty((t, h), dtype=out_dtype, device=x.device)
    _check(_LIB.vdamd_layer_norm_to(out.data_ptr(), x.data_ptr(), x.stride(0), None, 0,
                                    _f32_vec(weight, h, "weight").data_ptr(), _ptr(_f32_vec(bias, h, "bias")),
                                    float(eps), t, h, _dt(x), _dt(x), _DT[out_dtype], _stream()), "layer_norm_to")
    return out


def add_layer_norm(y: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                   eps: float, out_dtype: torch.dtype) -> torch.Tensor:
    t, h = y.shape
    assert residual.shape == (t, h) and residual.dtype == torch.float32 and residual.is_contiguous() and y.stride(1) == 1
    out = torch.empty((t, h), dtype=out_dtype, device=y.device)
    _check(_LIB.vdamd_layer_norm_to(out.data_ptr(), residual.data_ptr(), h, y.data_ptr(), y.stride(0),
                                    _f32_vec(weight, h, "weight").data_ptr(), _ptr(_f32_vec(bias, h, "bias")),
                                    float(eps), t, h, _DT[torch.float32], _dt(y), _DT[out_dtype], _stream()),
           "add_layer_norm")
    return out


DECAY_ATTENTION_MAX_DIM = 256


# ------------------------------------------------ recurrent mixers over prompt portions, 64 rows at a time
LINEAR_HEAD, LINEAR_CHANNEL, STATE_SPACE, DELTA_CHANNEL, DELTA_HEAD = range(5)
CHUNK_MAX_DIM = 128
CHUNK_MIN_ROWS = 48
CHUNK_SCRATCH_BYTES = 1 << 30


# Per recurrence, in us.  The chunked kernels: a call; a link of 64 rows of the longest sequence, and of 128 keys; per chunk and head
# the preparation of 128 keys, and the walk over them of 128 values, and of 128 values and 128 keys; the chunks that a sequence adds
# to its rows'.  The walk row by row: a call, a row of the longest sequence, a row and head, the same per 128 x 128 of the state, the
# rows that a sequence adds, and the power of (longest / average sequence) by which unequal ones leave the chip idle.  Fitted over
# 8000 to 12000 calls of each kind, one after the other from Python: 1 - 100 sequences, alike, unequal, prompts beside decoded rows, the
# longest of 48 rows and more, 2 - 64 heads, sizes 16 to 256, mild and strong decays (8 to 32 heads of 64 and 128 counting fivefold).
# Off by 9 to 18 % (root mean square), chunks of many sequences that fill their last one badly by up to 25.
CHUNK_COSTS = {LINEAR_HEAD: (18.6, 0.58, 1.71, 0.0204, 0.0236, 0.0419, 1.55, 3.7, 0.271, 0.00017, 0.00222, 3.7, 0.46),
               LINEAR_CHANNEL: (16.8, 0.58, 1.63, 0.0223, 0.0167, 0.0480, 1.47, 6.3, 0.230, 0.00002, 0.00208, 1.0, 0.65),
               STATE_SPACE: (17.8, 0.76, 1.26, 0.0166, 0.0241, 0.0357, 1.50, 4.3, 0.343, 0.00021, 0.00269, 4.2, 0.41),
               DELTA_CHANNEL: (24.3, 0.22, 2.80, 0.0480, 0.0130, 0.0533, 1.32, 16.2, 0.377, 0.00059, 0.00294, 7.1, 0.18),
               DELTA_HEAD: (20.9, 0.53, 2.34, 0.0392, 0.0314, 0.0287, 1.35, 14.3, 0.342, 0.00042, 0.00257, 7.0, 0.16)}


def _chunk_and_walk(kind: int, rows: int, seqs: int, longest: int, heads: int, dim: int, vdim: int) -> Tuple[float, float]:
    """Modelled times of the chunked kernels and of the walk row by row."""
    call, link, link_keys, prep, share, share_keys, seq, walk_call, row, row_head, row_area, walk_seq, unequal = CHUNK_COSTS[kind]
    keys, values = (0.5 if dim <= 64 else 1.0), max(vdim, 32) / 128
    chunks = (rows / 64 + seq * seqs) * heads
    chunked = call + chunks * prep * keys + math.hypot(longest / 64 * (link + link_keys * keys),
                                                       chunks * values * (share + share_keys * keys))
    lanes = 1 << max(dim - 1, 1).bit_length()                  # (the walk's keys: the next power of two)
    idle = min(max(longest * seqs / max(rows, 1), 1.0), 8.0) ** unequal
    return chunked, walk_call + math.hypot(longest * row, (rows + walk_seq * seqs) * heads * idle
                                           * (row_head + row_area * lanes * vdim / 16384))


@functools.lru_cache(maxsize=1024)              # (a step's layers ask with the same sizes)
def chunk_scan_profitable(kind: int, rows: int, seqs: int, max_rows: int, heads: int, dim: int, vdim: int,
                          aligned: bool = True) -> bool:
    """Whether ``seqs`` sequences with ``rows`` rows in all, at most ``max_rows`` in one (0: unknown), go through the chunked
    kernels (``aligned``: their rows can be read 16 bytes at a time), by the times of ``CHUNK_COSTS``.  Over the calls that those were
    fitted on, and 7300 others in graphs, the delta rule's choice is 0.4 to 0.7 % above the faster of the two on average, over 5 %
    above it in one call of 30 (58 prompts of 150 rows in chunks of 64, 16 heads: 343 / 323).  The walk row by row is a chain of dependent
    steps per row of the longest sequence, and bound by issue where many sequences run; a chunk of 64 rows costs a link of a shorter
    chain and its share of the chip, however few rows it holds and however small a head is (walk / chunks: 16 heads, dim 128, one prompt of 700 rows 298 / 63 us under the delta rule per channel,
    64 heads, 97 rows 93 / 46; 16 heads of 16 x 16, 58 prompts of 155 rows 110 / 151)."""
    longest = max_rows if max_rows > 0 else rows // max(seqs, 1)
    if dim > CHUNK_MAX_DIM or longest < CHUNK_MIN_ROWS:
        return False
    chunked, walk = _chunk_and_walk(kind, rows, seqs, longest, heads, dim, vdim)
    return chunked * (1.0 if aligned else 1.2) < walk


def _chunked(kind: int, x: torch.Tensor, rows: int, seqs: int, max_rows: int, heads: int, dim: int, vdim: int) -> bool:
    if 0 < max_rows < CHUNK_MIN_ROWS:              # (decoded rows: 0.7 us of Python beside the 13 of the whole call)
        return False
    aligned = x.stride(0) * x.element_size() % 16 == 0 and x.data_ptr() % 16 == 0
    return chunk_scan_profitable(kind, rows, seqs, max_rows, heads, dim, vdim, aligned)


def _chunk_workspace(kind: int, rows: int, seqs: int, heads: int, dim: int, vdim: int) -> Tuple[int, int, int]:
    """A bound on a step's chunks, the floats of workspace per head, and the heads taken at a time under
    ``CHUNK_SCRATCH_BYTES``."""
    chunks = (rows + 63 * min(seqs, rows)) // 64
    floats = int(_LIB.vdamd_chunk_scan_floats(kind, dim, vdim)) * chunks
    return chunks, floats, min(heads, max(1, CHUNK_SCRATCH_BYTES // (4 * floats)))


def chunk_scan_bytes(kind: int, rows: int, seqs: int, heads: int, dim: int, vdim: int) -> int:
    """What a recurrence over up to ``rows`` rows of up to ``seqs`` sequences allocates at most: workspace and result."""
    out = 4 * rows * heads * vdim
    if dim > CHUNK_MAX_DIM or rows < CHUNK_MIN_ROWS:
        return out
    _, floats, at_a_time = _chunk_workspace(kind, rows, max(seqs, 1), heads, dim, vdim)
    return out + 4 * floats * at_a_time


def chunk_columns(kind: int, rows: int, seqs: int, max_rows: int, heads: int, dim: int, vdim: int) -> int:
    """Columns of the state that a workgroup of the chunked kernels' walk has, 16 or 32.  With 32 a chunk takes longer, 3.8 against 3.0
    us under the delta rule, but the work in all is less: where the workgroups of 32 still give every compute unit one.  Delta rule
    over more than 64 keys: where 136 of them are busy on average until the longest sequence's end.  us at 32 / 16 columns, 8 heads of
    128 x 128, a decay per head: 7000 rows of five prompts alike (160 busy) 128 / 160, of five with one of 2420 (92) 176 / 145, of
    seven with one of 1200 (187) 118 / 136, 3000 rows of seven with one of 686 (140) 70 / 69; 260 calls of 8 to 32 heads agree to 2 %.
    64 keys, where two workgroups of 16 fit a compute unit, 32 heads of 128 columns, 4000 rows of two prompts (256) 132 / 113, of four
    (512) 97 / 99."""
    wide = -(-seqs * heads // 8) * 8 * -(-vdim // 32)
    if kind in (DELTA_CHANNEL, DELTA_HEAD):
        if dim <= 64:
            return 32 if wide >= 512 else 16
        return 32 if wide * rows >= 136 * seqs * max_rows and wide >= 136 else 16
    return 32 if wide >= 256 else 16


def _chunk_scan(kind: int, x, q_off: int, k_off: int, v_off: int, beta, dt, dt_bias, a_log, decay, d_skip, num_heads: int,
                groups: int, dim: int, vdim: int, state, slots, query_start_loc, seq_lens, silu: bool, eps: float,
                scale: float, max_rows: int) -> torch.Tensor:
    """One of the five recurrences over all sequences of a step (shapes checked by the caller).  The workspace (about 120 KB
    per chunk of 64 rows and head, the delta rule 150) is kept under ``CHUNK_SCRATCH_BYTES`` by taking the heads in turns."""
    t, b = x.shape[0], seq_lens.shape[0]
    out = torch.empty((t, num_heads * vdim), dtype=torch.float32, device=x.device)
    if t == 0 or b == 0:
        return out
    chunks, floats, heads = _chunk_workspace(kind, t, b, num_heads, dim, vdim)
    ws = torch.empty(heads * floats, dtype=torch.float32, device=x.device)
    for h0 in range(0, num_heads, heads):
        _check(_LIB.vdamd_chunk_scan(
            out.data_ptr(), kind, x.data_ptr(), x.stride(0), q_off, k_off, v_off, _ptr(beta),
            0 if beta is None else beta.stride(0), _ptr(dt), 0 if dt is None else dt.stride(0), _ptr(dt_bias), _ptr(a_log),
            _ptr(decay), _ptr(d_skip), ws.data_ptr(), chunks, state.data_ptr(), slots.data_ptr(),
            query_start_loc.data_ptr(), seq_lens.data_ptr(), b, num_heads, groups, dim, vdim, h0,
            min(heads, num_heads - h0), chunk_columns(kind, t, b, max_rows, min(heads, num_heads - h0), dim, vdim), int(silu),
            float(eps), float(scale), _dt(x), _stream()), "chunk_scan")
    return out


# The recurrences without a delta rule over segments, in us: a call, a chunk of 32 rows (fixed, and per 128 x 128 of the state),
# what a workgroup begins with.  Fitted over 16000 timings of 4500 calls of each kind like those of CHUNK_COSTS, whole and with cuts of 96
# to 480 rows, those of 8 to 32 heads of 64 and 128 counting fivefold: off by 10 to 11 % where the cut is the rule's (under a decay per
# channel where decays are mild: 32 strong ones in a row are multiplied out, at twice the time, which only the kernel sees).  Then what a
# chunk of 64 x 64 takes more where two workgroups share a compute unit, and the part of the others' modelled time below which segments
# are taken.
SEGMENT_COSTS = {LINEAR_HEAD: (1.6, 3.07, 3.87, 7.1, 1.1, 0.90), LINEAR_CHANNEL: (3.4, 2.37, 3.14, 5.4, 1.0, 0.98),
                 STATE_SPACE: (4.0, 2.59, 2.15, 5.5, 1.0, 0.96)}


@functools.lru_cache(maxsize=1024)              # (a step's layers ask with the same sizes)
def segment_rows(kind: int, rows: int, seqs: int, max_rows: int, heads: int, dim: int, vdim: int) -> int:
    """Rows at which sequences are cut into segments that run side by side (0: none is cut), or -1: the chunked kernels, whose
    preparation of all chunks at once leaves a sequence the shorter chain, or the walk row by row.  A cut is the one with which all
    segments run at a time, by an estimate of how many there are (half a segment more for each sequence), or 96 rows.  A time is between
    the chain of the longest segment and the share of the chip that all of them take.

    Over 1050 calls of 8 to 32 heads of 64 and 128, prompts of 1 to 24 sequences, the choice is above the fastest kernel and cut by
    1.5 % (linear attention), 1.0 (per channel) and 1.9 (state space) on average; 8, 1 and 2 of 350 calls each are over 5 % slower than
    without segments, at worst 1.14 times.  us without / with: 6007 rows of three prompts, 16 heads of 128 x 128, linear attention
    192 / 167; one prompt of 7000, 8 heads of 128 x 128, state space 237 / 74; 16 sequences of 473 rows in all, 64 heads of 96 x 96,
    114 / 59; 54 of 8964, 16 heads of 128 x 128, linear attention 298 / 214; 23 of 710, 64 heads of 32 x 64, per channel 26 / 34: not
    chosen."""
    longest = max_rows if max_rows > 0 else -(-rows // max(seqs, 1))
    if longest < CHUNK_MIN_ROWS or dim > CHUNK_MAX_DIM or vdim > 256:     # (wider: more scratch than the chunks' operands)
        return -1
    begin, fixed, area, over, shared, ahead = SEGMENT_COSTS[kind]
    limit = ahead * min(_chunk_and_walk(kind, rows, seqs, longest, heads, dim, vdim))
    dp, vp = 64 if dim <= 64 else 128, 64 if vdim <= 64 else -(-vdim // 128) * 128
    share = min(vp, 128) * dp / 16384              # of a workgroup in the largest state tile
    work = heads * max(vp // 128, 1) / (512 if share <= 0.25 else 256)           # of the workgroups that run at a time, a segment's
    chunk = (fixed + area * share) * (shared if share <= 0.25 else 1.0)

    def time(cut: int, segments: float) -> float:
        return begin + math.hypot(cut / 32 * chunk + over, ((rows / 32 + 0.8 * seqs) * chunk + segments * over) * work)
    best, choice = time(longest, seqs), 0
    others = (rows - longest) / max(seqs - 1, 1)
    room = 1.0 / work - 0.5 * seqs                 # segments of whole length that run at a time
    for cut in (96, max(96, int(rows / room / 32 + 1) * 32) if room > 0 else 96):
        if cut >= longest:
            continue
        segments = -(-longest // cut) + (seqs - 1) * (others / cut + 0.5)
        more = max(segments - seqs, 1.0)           # (of the pass over the states alone; their sums go through memory)
        cut_time = (time(cut, segments) + 3.3 + (cut / 32 * chunk * 0.07 + over) * math.hypot(1.0, more * work)
                    + segments * heads * dp * vp / 16384 * 0.052)
        if cut_time < best:
            best, choice = cut_time, cut
    return choice if best < limit else -1


def _segment_scan(kind: int, x, q_off: int, k_off: int, v_off: int, dt, dt_bias, a_log, decay, d_skip, num_heads: int,
                  groups: int, dim: int, vdim: int, state, slots, query_start_loc, seq_lens, silu: bool, scale: float,
                  max_rows: int) -> Optional[torch.Tensor]:
    """A recurrence without a delta rule over all sequences of a step (shapes checked by the caller) in segments; None where other
    kernels are to do it."""
    t, b, per = x.shape[0], seq_lens.shape[0], 16 // x.element_size()
    rows = segment_rows(kind, t, b, max_rows, num_heads, dim, vdim) if t and b else -1
    if rows < 0 or (x.stride(0) % per or x.data_ptr() % 16 or q_off % per or k_off % per or v_off % per or dim % 8 or vdim % 8
                    or (kind == LINEAR_CHANNEL and decay.data_ptr() % 16) or num_heads * vdim > 1 << 20):
        return None
    segments = b if rows == 0 else (t + (rows - 1) * min(b, t)) // rows
    floats = int(_LIB.vdamd_segment_scan_floats(num_heads, dim, vdim)) * segments if rows else 0
    # (no more than chunk_scan_bytes, however many heads at a time that counts; workgroups that a launch can have)
    if 8 * floats > CHUNK_SCRATCH_BYTES or num_heads > 65535 or segments * num_heads * -(-vdim // 128) >= 1 << 23:
        return None
    out = torch.empty((t, num_heads * vdim), dtype=torch.float32, device=x.device)
    ws = torch.empty(floats, dtype=torch.float32, device=x.device) if floats else None
    _check(_LIB.vdamd_segment_scan(
        out.data_ptr(), kind, x.data_ptr(), x.stride(0), q_off, k_off, v_off, _ptr(dt), 0 if dt is None else dt.stride(0),
        _ptr(dt_bias), _ptr(a_log), _ptr(decay), _ptr(d_skip), _ptr(ws), rows, segments, state.data_ptr(), slots.data_ptr(),
        query_start_loc.data_ptr(), seq_lens.data_ptr(), b, num_heads, groups, dim, vdim, int(silu), float(scale), _dt(x),
        _stream()), "segment_scan")
    return out


def decay_linear_attention(x: torch.Tensor, num_heads: int, dim: int, vdim: int, decay: torch.Tensor,
                           state: torch.Tensor, slots: torch.Tensor, query_start_loc: torch.Tensor,
                           seq_lens: torch.Tensor, silu: bool = True, max_query_len: int = 0,
                           scale: float = 1.0, chunked: Optional[bool] = None) -> torch.Tensor:
    """``chunked`` forces the chunked kernels, or the walk row by row (tests, benchmarks); None: by size, segments among them."""
    t = x.shape[0]
    n = seq_lens.numel()
    if dim > DECAY_ATTENTION_MAX_DIM:
        raise NotImplementedError(f"decayed linear attention with key size {dim} > {DECAY_ATTENTION_MAX_DIM}")
    assert x.stride(1) == 1 and x.shape[1] >= num_heads * (2 * dim + vdim)
    assert state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (num_heads, dim, vdim)
    assert slots.dtype == seq_lens.dtype == query_start_loc.dtype == torch.int32
    assert slots.numel() >= n and query_start_loc.numel() >= n + 1
    if decay.dim() == 2:                 # one per row, head and key channel
        assert decay.shape == (t, num_heads * dim) and decay.dtype == torch.float32 and decay.is_contiguous()
    elif scale != 1.0:
        raise NotImplementedError("a scale on the result needs decays per key channel")
    kind = LINEAR_CHANNEL if decay.dim() == 2 else LINEAR_HEAD
    if chunked or (chunked is None and not 0 < max_query_len < CHUNK_MIN_ROWS):
        qs = num_heads * dim
        rates = decay if decay.dim() == 2 else _f32_vec(decay, num_heads, "decay")
        if chunked is None:
            out = _segment_scan(kind, x, 0, qs, 2 * qs, None, None, None, rates, None, num_heads, num_heads, dim, vdim, state, slots,
                                query_start_loc, seq_lens, silu, scale, max_query_len)
            if out is not None:
                return out
        if chunked or _chunked(kind, x, t, n, max_query_len, num_heads, dim, vdim):
            return _chunk_scan(kind, x, 0, qs, 2 * qs, None, None, None, None, rates, None, num_heads, num_heads, dim, vdim,
                               state, slots, query_start_loc, seq_lens, silu, 0.0, scale, max_query_len)
    out = torch.empty((t, num_heads * vdim), dtype=torch.float32, device=x.device)
    if decay.dim() == 2:
        _check(_LIB.vdamd_channel_decay_attention(
            out.data_ptr(), x.data_ptr(), x.stride(0), decay.data_ptr(), state.data_ptr(), slots.data_ptr(),
            query_start_loc.data_ptr(), seq_lens.data_ptr(), n, num_heads, dim, vdim, float(scale), int(bool(silu)),
            int(max_query_len), _dt(x), _stream()), "channel_decay_attention")
        return out
    _check(_LIB.vdamd_decay_linear_attention(out.data_ptr(), x.data_ptr(), x.stride(0),
                                             _f32_vec(decay, num_heads, "decay").data_ptr(), state.data_ptr(),
                                             slots.data_ptr(), query_start_loc.data_ptr(), seq_lens.data_ptr(), n,
                                             num_heads, dim, vdim, int(bool(silu)), int(max_query_len), _dt(x),
                                             _stream()),
           "decay_linear_attention")
    return out


def gated_rms_norm(o: torch.Tensor, weight: torch.Tensor, gate: torch.Tensor, eps: float,
                   out_dtype: torch.dtype, group: int = 0, scale: float = 1.0, out=None,
                   silu: bool = False) -> torch.Tensor:
    t, n = o.shape
    assert o.dtype == torch.float32 and o.is_contiguous() and gate.shape == (t, n) and gate.stride(1) == 1
    group = int(group or 0)
    assert group == 0 or n % group == 0
    if out is None:
        out = torch.empty((t, n), dtype=out_dtype, device=o.device)
    assert out.dim() == 2 and out.shape == (t, n) and out.stride(1) == 1
    _check(_LIB.vdamd_gated_rms_norm(out.data_ptr(), out.stride(0), o.data_ptr(),
                                     _f32_vec(weight, group or n, "weight").data_ptr(), gate.data_ptr(), gate.stride(0),
                                     float(eps), t, n, group, float(scale), 1 if silu else 0, _dt(gate), _dt(out),
                                     _stream()),
           "gated_rms_norm")
    return out


def clamped_glu(h: torch.Tensor, limit: float, alpha: float) -> torch.Tensor:
    f = h.shape[-1] // 2
    h2 = h.reshape(-1, 2 * f)
    if h2.stride(1) != 1:
        h2 = h2.contiguous()
    out = torch.empty((h2.shape[0], f), dtype=h.dtype, device=h.device)
    _check(_LIB.vdamd_clamped_glu(out.data_ptr(), h2.data_ptr(), h2.stride(0), h2.shape[0], f, float(limit),
                                  float(alpha), _dt(h2), _stream()), "clamped_glu")
    return out.view(h.shape[:-1] + (f,))


def relu_squared(x: torch.Tensor) -> torch.Tensor:
    xc = x if x.is_contiguous() else x.contiguous()
    out = torch.empty_like(xc)
    _check(_LIB.vdamd_relu_squared(out.data_ptr(), xc.data_ptr(), xc.numel(), _dt(xc), _stream()), "relu_squared")
    return out


def low_rank_decay(a: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], tau: float) -> torch.Tensor:
    rows, rank = _rows2d(a, "a").shape
    c = weight.shape[0]
    assert weight.shape == (c, rank) and weight.dtype == a.dtype and weight.is_contiguous()
    out = torch.empty((rows, c), dtype=torch.float32, device=a.device)
    _check(_LIB.vdamd_low_rank_decay(out.data_ptr(), a.data_ptr(), a.stride(0), weight.data_ptr(),
                                     _ptr(_f32_vec(bias, c, "bias")), rows, c, rank, 1.0 / float(tau), _dt(a), _stream()),
           "low_rank_decay")
    return out


def weighted_relu_squared(h: torch.Tensor, topw: torch.Tensor, inv: torch.Tensor) -> torch.Tensor:
    rows, f = _rows2d(h, "h").shape
    slots = topw.numel()
    assert topw.dtype == torch.float32 and topw.is_contiguous() and rows >= slots
    assert inv.dtype == torch.int32 and inv.is_contiguous() and inv.numel() == slots
    out = torch.empty((rows, f), dtype=h.dtype, device=h.device)
    _check(_LIB.vdamd_weighted_relu_squared(out.data_ptr(), h.data_ptr(), h.stride(0), topw.data_ptr(), inv.data_ptr(), slots,
                                            f, _dt(h), _stream()), "weighted_relu_squared")
    return out


def latent_prep(q: torch.Tensor, nope: int, q_lat: torch.Tensor, latent: Optional[torch.Tensor],
                norm_weight: Optional[torch.Tensor], eps: float, inv_freq: torch.Tensor, rot_scale: float,
                positions: torch.Tensor, cache: Optional[torch.Tensor], slot_mapping: Optional[torch.Tensor],
                fragments: Optional[torch.Tensor] = None, interleaved: bool = False) -> torch.Tensor:
    """``fragments``: the V^T fragment cache ``[blocks, 1, rank / 16, block / 8, 16, 8]`` of the matrix-core latent
    attention kernel, written beside the rows when the layer keeps one."""
    t, h, qd = q.shape
    rank, rope = q_lat.shape[2], qd - nope
    half = inv_freq.numel()
    assert q.stride(2) == 1 and q_lat.stride(2) == 1 and q_lat.shape == (h, t, rank) and q_lat.dtype == q.dtype
    assert inv_freq.dtype == torch.float32 and inv_freq.is_contiguous() and 2 * half <= rope
    assert positions.dtype == torch.int32 and positions.numel() >= t
    out = torch.empty((t, h, rank + rope), dtype=q.dtype, device=q.device)
    write = latent is not None and cache is not None and slot_mapping is not None
    if write:
        assert latent.shape == (t, rank + rope) and latent.stride(1) == 1 and latent.dtype == q.dtype
        assert cache.is_contiguous() and cache.dtype == q.dtype and cache.shape[1] == 1 and cache.shape[3] == rank + rope
        assert slot_mapping.dtype == torch.int32 and slot_mapping.numel() >= t
        if fragments is not None and fragments.numel():
            bs = cache.shape[2]
            assert fragments.is_contiguous() and fragments.dtype == q.dtype and rank % 16 == 0 and bs % 8 == 0
            assert tuple(fragments.shape[1:]) == (1, rank // 16, bs // 8, 16, 8) and fragments.shape[0] == cache.shape[0]
        else:
            fragments = None
    else:
        fragments = None
    _check(_LIB.vdamd_latent_prep(
        out.data_ptr(), q.data_ptr(), q.stride(0), q.stride(1), nope, q_lat.data_ptr(), q_lat.stride(0),
        q_lat.stride(1), latent.data_ptr() if write else None, latent.stride(0) if write else 0,
        _f32_vec(norm_weight, rank, "norm_weight").data_ptr() if write else None, float(eps), inv_freq.data_ptr(),
        half, float(rot_scale), positions.data_ptr(), cache.data_ptr() if write else None, _ptr(fragments),
        slot_mapping.data_ptr() if write else None, t, h, rank, rope, cache.shape[2] if write else 8,
        1 if interleaved else 0, _dt(q), _stream()), "latent_prep")
    return out


def latent_row_attention(q: torch.Tensor, cache: torch.Tensor, block_table: torch.Tensor,
                         token_seq: Optional[torch.Tensor], seq_lens: torch.Tensor, scale: float, rank: int,
                         max_seq_len: int = 0, window: int = 0, sinks=None, gate=None) -> torch.Tensor:
    t, h, dk = q.shape
    assert q.is_contiguous() and cache.is_contiguous() and cache.dtype == q.dtype
    assert cache.shape[1] == 1 and cache.shape[3] == dk and 0 < rank <= dk
    assert block_table.dtype == torch.int32 and block_table.stride(1) == 1 and seq_lens.dtype == torch.int32
    assert seq_lens.numel() >= t and (token_seq is None or (token_seq.dtype == torch.int32 and token_seq.numel() >= t))
    assert token_seq is not None or block_table.shape[0] >= t
    out = torch.empty((t, h, rank), dtype=q.dtype, device=q.device)
    gate_stride = 0
    if gate is not None:
        assert gate.dim() == 2 and gate.shape[0] >= t and gate.shape[1] == h and gate.stride(1) == 1 and gate.dtype == q.dtype
        gate_stride = gate.stride(0)
    _check(_LIB.vdamd_latent_row_attention(out.data_ptr(), q.data_ptr(), cache.data_ptr(), block_table.data_ptr(),
                                           block_table.stride(0), None if token_seq is None else token_seq.data_ptr(),
                                           seq_lens.data_ptr(), float(scale), t, h, dk, rank, cache.shape[2],
                                           int(window), _ptr(_f32_vec(sinks, h, "sinks")), _ptr(gate), gate_stride,
                                           _dt(q), _stream()), "latent_row_attention")
    return out


def expert_epilogue(routed: torch.Tensor, x: torch.Tensor, topw: Optional[torch.Tensor], topi: Optional[torch.Tensor],
                    real_experts: int, shared: Optional[torch.Tensor], gate: Optional[torch.Tensor]) -> torch.Tensor:
    t, h = routed.shape
    assert routed.is_contiguous() and x.shape == (t, h) and x.stride(1) == 1 and x.dtype == routed.dtype
    k = 0
    if topw is not None:
        k = topw.shape[1]
        assert topw.dtype == torch.float32 and topi.dtype == torch.int32 and topw.is_contiguous() and topi.is_contiguous()
        assert topw.shape == topi.shape == (t, k)
    if shared is not None:
        assert shared.shape == (t, h) and shared.is_contiguous() and shared.dtype == routed.dtype
        assert gate is not None and gate.numel() == t and gate.dtype == routed.dtype
    out = torch.empty_like(routed)
    _check(_LIB.vdamd_expert_epilogue(out.data_ptr(), routed.data_ptr(), x.data_ptr(), x.stride(0), _ptr(topw),
                                      _ptr(topi), k, int(real_experts), _ptr(shared),
                                      None if shared is None else gate.data_ptr(),
                                      0 if shared is None else gate.stride(0), t, h, _dt(routed), _stream()),
           "expert_epilogue")
    return out



# ------------------------------------------------ fp32 residual stream with RMS norms, side inputs per token,
# ------------------------------------------------ convolution + activation, the gated delta rule
def _rows2d(t: torch.Tensor, name: str) -> torch.Tensor:
    assert t.dim() == 2 and t.stride(1) == 1 and t.is_cuda, f"{name}: rows of a 2-D tensor with unit column stride"
    return t


def _residual_rms(x, a, b, y, post_w, w, eps, out_dtype, offset, normed, post_scale: float = 1.0, z=None,
                  post_w2=None) -> torch.Tensor:
    rows, h = _rows2d(x, "x").shape
    adds = a is not None or y is not None
    if adds:
        assert x.dtype == torch.float32, "the residual stream is fp32"
    in_dt = _dt(x)
    for t, name in ((a, "a"), (b, "b"), (y, "y"), (z, "z")):
        if t is not None:
            assert _rows2d(t, name).shape == (rows, h)
            in_dt = _dt(t)
    for u, v in ((a, b), (a, y), (b, y), (y, z)):
        assert u is None or v is None or u.dtype == v.dtype
    assert b is None or a is not None
    assert z is None or y is not None
    out = torch.empty((rows, h), dtype=out_dtype, device=x.device)
    _check(_LIB.vdamd_residual_rms(
        out.data_ptr(), h, x.data_ptr(), x.stride(0), _ptr(a), 0 if a is None else a.stride(0), _ptr(b),
        0 if b is None else b.stride(0), _ptr(y), 0 if y is None else y.stride(0), _ptr(z), 0 if z is None else z.stride(0),
        _ptr(_f32_vec(post_w, h, "post_weight")) if y is not None else None,
        _ptr(_f32_vec(post_w2, h, "post_weight2")) if z is not None else None, _ptr(_f32_vec(w, h, "weight")),
        float(offset), float(eps), rows, h, 1 if normed else 0, _dt(x), in_dt, _DT[out_dtype],
        float(post_scale), _stream()), "residual_rms")
    return out


def rms_norm_to(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float, out_dtype: torch.dtype,
                offset: float = 0.0) -> torch.Tensor:
    lead = x.shape[:-1]
    x2 = x if x.dim() == 2 else x.reshape(-1, x.shape[-1])
    return _residual_rms(x2, None, None, None, None, weight, eps, out_dtype, offset, True).view(lead + (x.shape[-1],))


def add_rms_norm_to(residual, a, b, weight, eps: float, out_dtype, offset: float = 0.0, normed: bool = True):
    assert residual.is_contiguous()
    return _residual_rms(residual, a, b, None, None, weight, eps, out_dtype, offset, normed)


def norm_add_norm(y, post_weight, residual, next_weight, eps: float, out_dtype, next_offset: float = 0.0,
                  next_normed: bool = True, post_scale: float = 1.0, second=None, plain=None):
    assert residual.is_contiguous()
    z, w2 = second if second is not None else (None, None)
    return _residual_rms(residual, plain, None, y, post_weight, next_weight, eps, out_dtype, next_offset, next_normed,
                         post_scale, z, w2)


def gelu_mul_rows(g: torch.Tensor, table: torch.Tensor, ids: torch.Tensor, col: int) -> torch.Tensor:
    rows, n = _rows2d(g, "g").shape
    assert _rows2d(table, "table").dtype == g.dtype and 0 <= col and col + n <= table.shape[1]
    assert ids.dtype == torch.int32 and ids.numel() >= rows and ids.is_contiguous()
    out = torch.empty((rows, n), dtype=g.dtype, device=g.device)
    _check(_LIB.vdamd_gelu_mul_rows(out.data_ptr(), g.data_ptr(), g.stride(0), table.data_ptr(), table.stride(0),
                                    ids.data_ptr(), int(col), n, rows, table.shape[0], _dt(g), _stream()), "gelu_mul_rows")
    return out


def sigmoid_mul(o: torch.Tensor, gate: torch.Tensor, scale: float = 1.0, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    rows, n = _rows2d(o, "o").shape
    assert _rows2d(gate, "gate").shape == (rows, n) and gate.dtype == o.dtype
    if out is None:
        out = torch.empty((rows, n), dtype=o.dtype, device=o.device)
    assert _rows2d(out, "out").shape == (rows, n) and out.dtype == o.dtype
    _check(_LIB.vdamd_sigmoid_mul(out.data_ptr(), out.stride(0), o.data_ptr(), o.stride(0), gate.data_ptr(),
                                  gate.stride(0), float(scale), rows, n, _dt(o), _stream()), "sigmoid_mul")
    return out


def gelu(x: torch.Tensor, tanh: bool) -> torch.Tensor:
    xc = x if x.is_contiguous() else x.contiguous()
    out = torch.empty_like(xc)
    _check(_LIB.vdamd_gelu(out.data_ptr(), xc.data_ptr(), xc.numel(), 1 if tanh else 0, _dt(xc), _stream()), "gelu")
    return out


def short_conv_act(x, channels: int, conv_weight, state, slots, query_start_loc, seq_lens, token_seq, positions,
                   silu: bool, has_prefill: bool = True, bias=None, residual: bool = False,
                   in_bias=None) -> torch.Tensor:
    t = _rows2d(x, "x").shape[0]
    c, taps = int(channels), conv_weight.shape[0]
    r = max(taps - 1, 1)
    b = seq_lens.shape[0]
    assert x.shape[1] >= c and conv_weight.shape == (taps, c) and conv_weight.dtype == x.dtype and conv_weight.is_contiguous()
    assert 1 <= taps <= CONV_MAX_TAPS
    assert state is not None and state.dtype == x.dtype and state.is_contiguous() and state.shape[1:] == (r, c), \
        (None if state is None else state.shape, (r, c))
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1 and positions.shape[0] >= t
    assert token_seq is None or token_seq.shape[0] >= t
    assert token_seq is not None or t <= b, "rows without a sequence"
    assert int(state.shape[0]) > 0
    out = torch.empty((t, c), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_short_conv_act(
        out.data_ptr(), c, x.data_ptr(), x.stride(0), conv_weight.data_ptr(), state.data_ptr(),
        _i32(slots, "slots").data_ptr(), _i32(query_start_loc, "query_start_loc").data_ptr(),
        _i32(seq_lens, "seq_lens").data_ptr(), _ptr(_i32(token_seq, "token_seq")),
        _i32(positions, "positions").data_ptr(), t, b, c, taps, 1 if silu else 0, 1 if has_prefill else 0,
        _ptr(_f32_vec(bias, c, "bias")), 1 if residual else 0, _ptr(_f32_vec(in_bias, c, "in_bias")), _dt(x), _stream()),
        "short_conv_act")
    return out


def gated_delta_rule(x, num_heads: int, num_qk_heads: int, dim: int, vdim: int, beta, dt, dt_bias, a_log, state, slots,
                     query_start_loc, seq_lens, norm_eps: float = 1e-6, max_query_len: int = 0,
                     parts: int = 0, chunked: Optional[bool] = None) -> torch.Tensor:
    """``max_query_len`` (0: unknown) only helps the kernel choose its tiling; ``parts`` forces one of the row by row walk,
    ``chunked`` the chunked kernels or the walk (tests, benchmarks).
    ``dt[T, H]``: one decay per head."""
    t = _rows2d(x, "x").shape[0]
    h, g = int(num_heads), int(num_qk_heads)
    b = seq_lens.shape[0]
    assert h % g == 0 and 0 < dim <= 256 and x.shape[1] >= 2 * g * dim + h * vdim
    assert _rows2d(beta, "beta").shape[0] >= t and beta.shape[1] == h and beta.dtype == x.dtype
    per_head = dt.shape[1] == h
    assert _rows2d(dt, "dt").shape[0] >= t and (per_head or dt.shape[1] == h * dim) and dt.dtype == x.dtype
    assert state is not None and state.dtype == torch.float32 and state.is_contiguous()
    assert tuple(state.shape[1:]) == (h, dim, vdim), (tuple(state.shape), (h, dim, vdim))
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1
    kind = DELTA_HEAD if per_head else DELTA_CHANNEL
    if (not parts and _chunked(kind, x, t, b, max_query_len, h, dim, vdim)) if chunked is None else chunked:
        return _chunk_scan(kind, x, 0, g * dim, 2 * g * dim, beta, dt,
                           _f32_vec(dt_bias, dt.shape[1], "dt_bias"), _f32_vec(a_log, h, "a_log"), None, None, h, g, dim, vdim,
                           state, _i32(slots, "slots"), _i32(query_start_loc, "query_start_loc"), _i32(seq_lens, "seq_lens"),
                           False, norm_eps, 1.0, max_query_len)
    out = torch.empty((t, h * vdim), dtype=torch.float32, device=x.device)
    if max_query_len == 1 and not parts and dim <= 128 and vdim % 4 == 0 and state.data_ptr() % 16 == 0 and b <= 65535:
        _check(_LIB.vdamd_delta_rule_rows(
            out.data_ptr(), x.data_ptr(), x.stride(0), beta.data_ptr(), beta.stride(0), dt.data_ptr(), dt.stride(0),
            _f32_vec(dt_bias, dt.shape[1], "dt_bias").data_ptr(), _f32_vec(a_log, h, "a_log").data_ptr(), state.data_ptr(),
            _i32(slots, "slots").data_ptr(), _i32(query_start_loc, "query_start_loc").data_ptr(),
            _i32(seq_lens, "seq_lens").data_ptr(), b, h, g, dim, vdim, int(per_head), float(norm_eps), _dt(x), _stream()),
            "delta_rule_rows")
        return out
    dev = x.device
    qn = torch.empty((t, g, dim), dtype=torch.float32, device=dev)
    kn = torch.empty((t, g, dim), dtype=torch.float32, device=dev)
    decay = None if per_head else torch.empty((t, h, dim), dtype=torch.float32, device=dev)
    # sigmoid(beta) | k.q of the head's group (| the head's decay)
    bsig = torch.empty((t, 3 if per_head else 2, h), dtype=torch.float32, device=dev)
    _check(_LIB.vdamd_delta_rule_prep(
        qn.data_ptr(), kn.data_ptr(), _ptr(decay), bsig.data_ptr(), x.data_ptr(), x.stride(0), beta.data_ptr(),
        beta.stride(0), dt.data_ptr(), dt.stride(0), _f32_vec(dt_bias, dt.shape[1], "dt_bias").data_ptr(),
        _f32_vec(a_log, h, "a_log").data_ptr(), t, h, g, dim, float(norm_eps), _dt(x), _stream()), "delta_rule_prep")
    _check(_LIB.vdamd_gated_delta_rule(
        out.data_ptr(), x.data_ptr(), x.stride(0), 2 * g * dim, qn.data_ptr(), kn.data_ptr(), _ptr(decay),
        bsig.data_ptr(), state.data_ptr(), _i32(slots, "slots").data_ptr(),
        _i32(query_start_loc, "query_start_loc").data_ptr(), _i32(seq_lens, "seq_lens").data_ptr(), b, h, g, dim, vdim,
        int(max_query_len), int(parts), _dt(x), _stream()), "gated_delta_rule")
    return out


# ------------------------------------------------ selective state-space scan, gate in front of a grouped norm,
# ------------------------------------------------ q / k normed over all heads with values = keys, mixed head weights
def selective_scan(x, dt, num_heads: int, groups: int, vdim: int, n_state: int, a_log, dt_bias, d_skip, state, slots,
                   query_start_loc, seq_lens, max_query_len: int = 0, chunked: Optional[bool] = None) -> torch.Tensor:
    """``max_query_len`` (0: unknown) only helps choose the kernel; ``chunked`` forces the chunked kernels, or the walk row by row
    (tests, benchmarks); None: by size, segments among them."""
    t = _rows2d(x, "x").shape[0]
    h, g, n = int(num_heads), int(groups), int(n_state)
    b = seq_lens.shape[0]
    assert h % g == 0 and 0 < n <= 256 and x.shape[1] >= h * vdim + 2 * g * n
    assert _rows2d(dt, "dt").shape[0] >= t and dt.shape[1] >= h and dt.dtype == x.dtype
    assert state is not None and state.dtype == torch.float32 and state.is_contiguous()
    assert tuple(state.shape[1:]) == (h, n, vdim), (tuple(state.shape), (h, n, vdim))
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1
    if chunked or (chunked is None and not 0 < max_query_len < CHUNK_MIN_ROWS):
        inner = h * vdim
        mine = (_f32_vec(dt_bias, h, "dt_bias"), _f32_vec(a_log, h, "a_log"), None, _f32_vec(d_skip, h, "d_skip"), h, g, n, int(vdim),
                state, _i32(slots, "slots"), _i32(query_start_loc, "query_start_loc"), _i32(seq_lens, "seq_lens"), False)
        if chunked is None:
            out = _segment_scan(STATE_SPACE, x, inner + g * n, inner, 0, dt, *mine, 1.0, max_query_len)
            if out is not None:
                return out
        if chunked or _chunked(STATE_SPACE, x, t, b, max_query_len, h, n, int(vdim)):
            return _chunk_scan(STATE_SPACE, x, inner + g * n, inner, 0, None, dt, *mine, 0.0, 1.0, max_query_len)
    out = torch.empty((t, h * vdim), dtype=torch.float32, device=x.device)
    _check(_LIB.vdamd_selective_scan(
        out.data_ptr(), x.data_ptr(), x.stride(0), dt.data_ptr(), dt.stride(0), _f32_vec(a_log, h, "a_log").data_ptr(),
        _f32_vec(dt_bias, h, "dt_bias").data_ptr(), _ptr(_f32_vec(d_skip, h, "d_skip")), state.data_ptr(),
        _i32(slots, "slots").data_ptr(), _i32(query_start_loc, "query_start_loc").data_ptr(),
        _i32(seq_lens, "seq_lens").data_ptr(), b, h, g, n, int(vdim), int(max_query_len), _dt(x), _stream()),
        "selective_scan")
    return out


def act_gate_group_norm(y: torch.Tensor, gate: torch.Tensor, weight: torch.Tensor, eps: float, group: int,
                        out_dtype: torch.dtype) -> torch.Tensor:
    t, n = y.shape
    group = int(group) or n
    assert y.dtype == torch.float32 and y.is_contiguous() and n % group == 0
    assert _rows2d(gate, "gate").shape[0] >= t and gate.shape[1] >= n and gate.dtype == out_dtype
    out = torch.empty((t, n), dtype=out_dtype, device=y.device)
    _check(_LIB.vdamd_act_gate_group_norm(out.data_ptr(), y.data_ptr(), gate.data_ptr(), gate.stride(0),
                                          _f32_vec(weight, n, "weight").data_ptr(), float(eps), t, n, group,
                                          _dt(out), _stream()), "act_gate_group_norm")
    return out


def joint_norm_cache(x, num_heads: int, num_kv_heads: int, dim: int, q_norm, k_norm, eps: float, positions,
                     temp_coef: float, temp_every: int, k_cache, v_cache, slot_mapping) -> torch.Tensor:
    t = _rows2d(x, "x").shape[0]
    h, g, d = int(num_heads), int(num_kv_heads), int(dim)
    assert x.shape[1] >= (h + g) * d and positions.shape[0] >= t
    bs = 0
    if k_cache is not None:
        bs = k_cache.shape[2]
        assert k_cache.dtype == v_cache.dtype == x.dtype and k_cache.is_contiguous() and v_cache.is_contiguous()
        assert tuple(k_cache.shape[1:]) == (g, bs, d) and bs % 8 == 0
        assert tuple(v_cache.shape) == (k_cache.shape[0], g, bs // 8, d, 8)
        assert slot_mapping.shape[0] >= t
    q = torch.empty((t, h, d), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_joint_norm_cache(
        q.data_ptr(), x.data_ptr(), x.stride(0), _f32_vec(q_norm, h * d, "q_norm").data_ptr(),
        _f32_vec(k_norm, g * d, "k_norm").data_ptr(), float(eps), _i32(positions, "positions").data_ptr(),
        float(temp_coef), int(temp_every), _ptr(k_cache), _ptr(v_cache),
        _ptr(_i32(slot_mapping, "slot_mapping") if k_cache is not None else None), t, h, g, d, int(bs), _dt(x),
        _stream()), "joint_norm_cache")
    return q


def mix_heads(o: torch.Tensor, talk: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    t, h, g, dv = o.shape
    assert o.dtype == torch.float32 and o.is_contiguous() and h % g == 0
    out = torch.empty((t, h * dv), dtype=out_dtype, device=o.device)
    _check(_LIB.vdamd_mix_heads(out.data_ptr(), o.data_ptr(), _f32_vec(talk, h * h, "talk").data_ptr(), t, h, g, dv,
                                _dt(out), _stream()), "mix_heads")
    return out


# ------------------------------------------------ rotation in front of a head norm, a selective scan per channel, a
# ------------------------------------------------ gated linear unit recurrence
def rotate_norm_cache(x, num_heads: int, num_kv_heads: int, dim: int, vdim: int, inv_freq, rot_scale: float,
                      interleaved: bool, eps: float, q_norm, k_norm, positions, k_cache, v_cache,
                      slot_mapping, normed: bool = True, bias=None) -> torch.Tensor:
    t = _rows2d(x, "x").shape[0]
    h, g, d, dv = int(num_heads), int(num_kv_heads), int(dim), int(vdim)
    assert x.shape[1] >= (h + g) * d + g * dv and positions.shape[0] >= t and d <= UNIT_MAX_WIDTH
    assert (h % g == 0) if g else k_cache is None
    half = 0 if inv_freq is None else int(inv_freq.numel())
    assert 2 * half <= d
    bs = 0
    if k_cache is not None:
        bs = k_cache.shape[2]
        assert k_cache.dtype == v_cache.dtype == x.dtype and k_cache.is_contiguous() and v_cache.is_contiguous()
        assert tuple(k_cache.shape[1:]) == (g, bs, d) and bs % 8 == 0
        assert tuple(v_cache.shape) == (k_cache.shape[0], g, bs // 8, dv, 8)
        assert slot_mapping.shape[0] >= t
    q = torch.empty((t, h, d), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_rotate_norm_cache(
        q.data_ptr(), x.data_ptr(), x.stride(0), _ptr(_f32_vec(inv_freq, half, "inv_freq")) if half else None, half,
        float(rot_scale), 1 if interleaved else 0, float(eps), _ptr(_f32_vec(q_norm, d, "q_norm")),
        _ptr(_f32_vec(k_norm, d, "k_norm")), _ptr(_f32_vec(bias, (h + g) * d + g * dv, "bias")),
        _i32(positions, "positions").data_ptr(), _ptr(k_cache), _ptr(v_cache),
        _ptr(_i32(slot_mapping, "slot_mapping") if k_cache is not None else None), t, h, g, d, dv, int(bs),
        1 if normed else 0, _dt(x), _stream()), "rotate_norm_cache")
    return q


def gelu_and_mul(x: torch.Tensor, tanh: bool = True) -> torch.Tensor:
    f = x.shape[-1] // 2
    x2 = x.reshape(-1, 2 * f)
    if x2.stride(1) != 1:
        x2 = x2.contiguous()
    out = torch.empty((x2.shape[0], f), dtype=x.dtype, device=x.device)
    _check(_LIB.vdamd_gelu_and_mul(out.data_ptr(), x2.data_ptr(), x2.stride(0), x2.shape[0], f, 1 if tanh else 0, _dt(x2),
                                   _stream()), "gelu_and_mul")
    return out.view(x.shape[:-1] + (f,))


def channel_scan(u, dt, bc, n_state: int, a_log, dt_bias, d_skip, gate, state, slots, query_start_loc, seq_lens,
                 max_query_len: int = 0) -> torch.Tensor:
    """``max_query_len`` (0: unknown) only helps the kernel choose its launch; 1 must be true."""
    t, c = _rows2d(u, "u").shape
    n, b = int(n_state), seq_lens.shape[0]
    if not 0 < n <= 256:
        raise NotImplementedError(f"a selective scan with {n} states per channel (at most 256)")
    assert _rows2d(dt, "dt").shape[0] >= t and dt.shape[1] == c and dt.dtype in (u.dtype, torch.float32)
    assert _rows2d(bc, "bc").shape[0] >= t and bc.shape[1] >= 2 * n and bc.dtype == u.dtype
    if gate is not None:
        assert _rows2d(gate, "gate").shape[0] >= t and gate.shape[1] == c and gate.dtype == u.dtype
    assert state is not None and state.dtype == torch.float32 and state.is_contiguous()
    assert tuple(state.shape[1:]) == (c, n), (tuple(state.shape), (c, n))
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1
    assert max_query_len != 1 or t <= b
    out = torch.empty((t, c), dtype=u.dtype, device=u.device)
    _check(_LIB.vdamd_channel_scan(
        out.data_ptr(), u.data_ptr(), u.stride(0), dt.data_ptr(), dt.stride(0), bc.data_ptr(), bc.stride(0), _ptr(gate),
        0 if gate is None else gate.stride(0), _f32_vec(a_log, c * n, "a_log").data_ptr(),
        _ptr(_f32_vec(dt_bias, c, "dt_bias")), _ptr(_f32_vec(d_skip, c, "d_skip")), state.data_ptr(),
        _i32(slots, "slots").data_ptr(), _i32(query_start_loc, "query_start_loc").data_ptr(),
        _i32(seq_lens, "seq_lens").data_ptr(), b, c, n, int(max_query_len), _dt(u), _dt(dt), _stream()), "channel_scan")
    return out


def _block_gates(u, ra, ra_bias, ri, ri_bias, rate, a, drive, out, gate, gate_bias, state, slots, seq_lens) -> None:
    t, w = _rows2d(u, "u").shape
    n = ra.shape[1]
    assert u.is_contiguous() and ra.is_contiguous() and ri.is_contiguous() and ra.dtype == ri.dtype == u.dtype
    assert ra.shape == ri.shape == (w // n, n, n) and w % n == 0
    _check(_LIB.vdamd_block_gates(
        _ptr(a), _ptr(drive), u.data_ptr(), ra.data_ptr(), _f32_vec(ra_bias, w, "ra_bias").data_ptr(), ri.data_ptr(),
        _f32_vec(ri_bias, w, "ri_bias").data_ptr(), _f32_vec(rate, w, "rate").data_ptr(), _ptr(out), _ptr(gate),
        0 if gate is None else gate.stride(0), _ptr(_f32_vec(gate_bias, w, "gate_bias")), _ptr(state), _ptr(slots),
        _ptr(seq_lens), t, w, n, _dt(u), _stream()), "block_gates")


def block_gates(u, ra, ra_bias, ri, ri_bias, rate):
    a = torch.empty(u.shape, dtype=torch.float32, device=u.device)
    drive = torch.empty_like(a)
    _block_gates(u, ra, ra_bias, ri, ri_bias, rate, a, drive, None, None, None, None, None, None)
    return a, drive


def gated_unit_scan(a, drive, gate, gate_bias, state, slots, query_start_loc, seq_lens,
                    max_query_len: int = 0) -> torch.Tensor:
    t, w = a.shape
    b = seq_lens.shape[0]
    assert a.dtype == drive.dtype == torch.float32 and a.is_contiguous() and drive.is_contiguous() and drive.shape == a.shape
    assert _rows2d(gate, "gate").shape[0] >= t and gate.shape[1] == w
    assert state is not None and state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (w,)
    assert slots.shape[0] == b and query_start_loc.shape[0] >= b + 1
    out = torch.empty((t, w), dtype=gate.dtype, device=a.device)
    _check(_LIB.vdamd_gated_unit_scan(
        out.data_ptr(), a.data_ptr(), drive.data_ptr(), gate.data_ptr(), gate.stride(0),
        _ptr(_f32_vec(gate_bias, w, "gate_bias")), state.data_ptr(), _i32(slots, "slots").data_ptr(),
        _i32(query_start_loc, "query_start_loc").data_ptr(), _i32(seq_lens, "seq_lens").data_ptr(), b, w,
        int(max_query_len), _dt(gate), _stream()), "gated_unit_scan")
    return out


def gated_unit_step(u, ra, ra_bias, ri, ri_bias, rate, gate, gate_bias, state, slots, query_start_loc, seq_lens,
                    max_query_len: int = 0) -> torch.Tensor:
    t, w = u.shape
    if (max_query_len == 1 and t == seq_lens.shape[0] and gate.stride(0) % 4 == 0 and gate.data_ptr() % 8 == 0
            and _LIB.vdamd_block_gates_mfma_ok(int(ra.shape[1]), _dt(u))):
        # every row is its sequence's only one: gates, state and output gate in one launch
        assert state is not None and state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (w,)
        assert _rows2d(gate, "gate").shape == (t, w) and gate.dtype == u.dtype and slots.shape[0] == t
        out = torch.empty((t, w), dtype=u.dtype, device=u.device)
        _block_gates(u, ra, ra_bias, ri, ri_bias, rate, None, None, out, gate, gate_bias, state, _i32(slots, "slots"),
                     _i32(seq_lens, "seq_lens"))
        return out
    a, drive = block_gates(u, ra, ra_bias, ri, ri_bias, rate)
    return gated_unit_scan(a, drive, gate, gate_bias, state, slots, query_start_loc, seq_lens, max_query_len)
