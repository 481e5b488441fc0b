"""Fused LTX-2.3 DiT block ops on MI355X: drop-in for `ltx_serve/triton_ltx_ops.py`.

Every public function keeps the name, signature, argument meaning, output
allocation and guard behaviour of plugyawn/opengenie's
`ltx_serve/triton_ltx_ops.py` (file:line cited per function), so the denoise
loop can call this module in its place. When an input passes the op's guard,
the op runs as a hand-written gfx950 HIP kernel from libopengenie_amd.so on
torch's current stream; nothing synchronises. When the guard fails, the op
evaluates the reference's own torch expression on the tensors' device, as the
reference does. The library being absent is not a guard failure: a tensor
that would take the HIP path raises `LibraryMissing`. Setting
OPENGENIE_AMD_STRICT=1 makes a guard failure on GPU tensors raise instead of
falling back (the parity tests run that way).

Rounding contract: the HIP kernels compute in float32 and round to bf16
exactly where torch, evaluating the reference's torch expression, would hold a
bf16 result; FP8 codes equal torch's conversion of the same expression.
"""

from __future__ import annotations

import os
import weakref

import torch

from . import _lib

__all__ = [
    "fused_adazero",
    "fused_adazero_from_ada",
    "fused_adazero_from_ada_fp8",
    "fused_adaln_affine_from_ada",
    "fused_fp8_quantize_e4m3",
    "fused_gelu_tanh_fp8_quantize_e4m3",
    "fused_bias_add_bf16",
    "fused_residual_gate_bias_from_ada",
    "fused_fp8_quantize_e4m3_per_head_4d",
    "fused_video_qk_rmsnorm_rope",
    "fused_video_qkv_rmsnorm_rope_pack",
    "fused_video_qk_rmsnorm_rope_separate",
    "fused_video_qk_bias_rmsnorm_rope",
    "qk_rmsnorm",
    "fused_residual_gate_bf16",
    "fused_head_gate_mul_bf16",
    "fused_residual_gate_from_ada",
    "fused_residual_gate_adazero_from_ada",
    "fused_mul_from_ada",
    "fp8_linear_from_quantized_e4m3",
    "fp8_linear_without_bias",
    "fp8_linear_forward",
    "fp8_scaled_mm",
    "fp8_qkv_from_shared_quantized_input",
    "fp8_qkv_from_grouped_mm",
    "fp8_qkv_from_quantized_e4m3",
    "fp8_qk_from_grouped_mm",
    "fp8_kv_from_grouped_mm",
    "fp8_qkv_from_packed_linear",
    "fp8_qkv_from_packed_requant",
    "collect_video_qkv_packed_linear_stats",
    "collect_video_qkv_packed_requant_stats",
    "collect_video_qkv_grouped_mm_stats",
    "collect_video_qk_grouped_mm_stats",
    "reset_video_qkv_grouped_mm_stats",
    "reset_video_qk_grouped_mm_stats",
    "reset_video_qkv_packed_stats",
    "set_frozen_fp8_scales",
    "frozen_fp8_scales",
]

_FP8 = torch.float8_e4m3fn
_FP8_MAX = 448.0
_DT_CODES = {torch.bfloat16: _lib.DT_BF16, torch.float16: _lib.DT_F16, torch.float32: _lib.DT_F32}

# --------------------------------------------------------------------------
# bookkeeping (mirrors the reference's module counters, :1992-2034)
# --------------------------------------------------------------------------
_VIDEO_ADA_VALUES_CALLS = 0
_AUDIO_ADA_VALUES_CALLS = 0
_VIDEO_TEXT_ADALN_CALLS = 0
_HIP_CALLS: dict[str, int] = {}

# Production residual mode of the reference worker (triton_ltx_ops.py
# :1977-1981 as pinned by remote_official_worker.py:938-972).
_BLOCK_RESIDUAL_MODE = "triton_simple_bf16_round"


def _increment_ada_counter(counter: str) -> None:
    """:2008-2015"""
    global _VIDEO_ADA_VALUES_CALLS, _AUDIO_ADA_VALUES_CALLS, _VIDEO_TEXT_ADALN_CALLS
    if counter == "video":
        _VIDEO_ADA_VALUES_CALLS += 1
    elif counter == "audio":
        _AUDIO_ADA_VALUES_CALLS += 1
    elif counter == "video_text":
        _VIDEO_TEXT_ADALN_CALLS += 1


def collect_video_ada_values_calls() -> int:
    return _VIDEO_ADA_VALUES_CALLS


def collect_audio_ada_values_calls() -> int:
    return _AUDIO_ADA_VALUES_CALLS


def collect_video_text_adaln_calls() -> int:
    return _VIDEO_TEXT_ADALN_CALLS


def collect_hip_calls() -> dict[str, int]:
    """How many times each op took the HIP kernel path in this process."""
    return dict(_HIP_CALLS)


def reset_hip_calls() -> None:
    _HIP_CALLS.clear()


def set_block_residual_mode(mode: str) -> None:
    """Selects `_simple_residual_gate`'s arithmetic (:1955-1960)."""
    global _BLOCK_RESIDUAL_MODE
    if mode not in {"addcmul", "addcmul_simple", "triton_bf16_round", "triton_simple_bf16_round", "simple"}:
        raise ValueError(f"unknown residual mode: {mode}")
    _BLOCK_RESIDUAL_MODE = mode


def _hip(name: str) -> None:
    _HIP_CALLS[name] = _HIP_CALLS.get(name, 0) + 1


def _strict() -> bool:
    return os.environ.get("OPENGENIE_AMD_STRICT", "0") not in ("", "0")


def _fallback(name: str, *tensors: torch.Tensor) -> None:
    """Called when a guard fails. Under OPENGENIE_AMD_STRICT a GPU input raises."""
    if _strict() and any(isinstance(t, torch.Tensor) and t.is_cuda for t in tensors):
        raise RuntimeError(f"{name}: input not supported by the HIP kernel (strict mode)")


def _dt(t: torch.Tensor) -> int:
    return _lib.DT_BF16 if t.dtype == torch.bfloat16 else _lib.DT_F32


def _xdt(t: torch.Tensor) -> int:
    """dtype code of a 16-bit activation (bf16 or fp16)."""
    return _lib.DT_F16 if t.dtype == torch.float16 else _lib.DT_BF16


def _any_dt(t: torch.Tensor) -> int:
    """dtype code of a bf16, fp16 or float32 tensor."""
    return _DT_CODES[t.dtype]


def _stream(t: torch.Tensor) -> int:
    """The raw handle of the current stream of t's device: what
    torch.cuda.current_stream(t.device).cuda_stream holds, without the Stream
    object made on each call."""
    return torch._C._cuda_getCurrentRawStream(t.get_device())


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def _aligned(t: torch.Tensor, nbytes: int = 16) -> bool:
    """The C ABI's pointer precondition for a tensor it reads with 128-bit
    (or wider) vectors. A contiguous view at an odd storage offset passes the
    reference's guards but not this one, so it takes the torch path instead
    of an argument error from the library."""
    return t.data_ptr() % nbytes == 0


# --------------------------------------------------------------------------
# torch reference paths (the reference's fallbacks)
# --------------------------------------------------------------------------
def _torch_ada_values_from_table(
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    batch_size: int,
    tokens: int,
    cols: int,
    *indices: int,
) -> tuple[torch.Tensor, ...]:
    """:983-998"""
    ts_view = timestep.reshape(batch_size, timestep.shape[1], scale_shift_table.shape[0], -1)
    if ts_view.shape[1] != tokens or ts_view.shape[-1] != cols:
        raise ValueError(
            f"Unexpected Ada timestep shape {tuple(timestep.shape)} for x shape "
            f"({batch_size}, {tokens}, {cols}) and table {tuple(scale_shift_table.shape)}"
        )
    table = scale_shift_table.to(device=timestep.device, dtype=timestep.dtype)
    return tuple(table[i].view(1, 1, cols) + ts_view[:, :, i, :] for i in indices)


def _torch_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, eps, cos, sin):
    """:958-973, with split RoPE written out as the reference's test restates it
    (tests/test_triton_ltx_ops.py:232-249); ltx_core is not a dependency."""
    q = torch.nn.functional.rms_norm(q, (q.shape[-1],), weight=q_weight, eps=eps)
    k = torch.nn.functional.rms_norm(k, (k.shape[-1],), weight=k_weight, eps=eps)
    return _torch_split_rope(q, cos, sin), _torch_split_rope(k, cos, sin)


def _torch_split_rope(x, cos, sin):
    b, n, dim = x.shape
    heads = cos.shape[1]
    hd = dim // heads
    half = hd // 2
    xh = x.reshape(b, n, heads, hd).transpose(1, 2)
    first, second = xh[..., :half], xh[..., half:]
    out = torch.cat([first * cos - second * sin, second * cos + first * sin], dim=-1)
    return out.transpose(1, 2).reshape(b, n, dim)


def _torch_fp8_quantize_e4m3_per_head_4d(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """:976-980"""
    scale = x.float().abs().amax(dim=(1, 3)).clamp_min(1e-12) / _FP8_MAX
    q = torch.clamp(x.float() / scale[:, None, :, None], -_FP8_MAX, _FP8_MAX).to(_FP8)
    return q, scale.to(torch.float32).contiguous()


def _simple_residual_gate(x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """:1955-1960"""
    if _BLOCK_RESIDUAL_MODE in {"triton_bf16_round", "triton_simple_bf16_round"}:
        return fused_residual_gate_bf16(x, y, gate)
    if _BLOCK_RESIDUAL_MODE in {"addcmul", "addcmul_simple"}:
        return torch.addcmul(x, y, gate)
    return x + y * gate


# --------------------------------------------------------------------------
# guards (same conditions as the reference; "triton is None" has no
# counterpart: a missing library raises instead of falling back)
# --------------------------------------------------------------------------
def _can_use_ada_from_table(x: torch.Tensor, scale_shift_table: torch.Tensor, timestep: torch.Tensor) -> bool:
    """:1001-1018, plus the HIP kernels' own needs: x 16-byte aligned and at
    most 65535 batches (one grid row per batch)."""
    if not x.is_cuda or not x.is_contiguous() or x.dtype != torch.bfloat16:
        return False
    shape, table_shape, ts_shape = x.shape, scale_shift_table.shape, timestep.shape
    if len(shape) != 3 or shape[2] not in (2048, 4096):
        return False
    if not _aligned(x) or shape[0] > 65535:
        return False
    if not scale_shift_table.is_cuda or scale_shift_table.dtype not in (torch.bfloat16, torch.float32):
        return False
    if len(table_shape) != 2 or table_shape[1] != shape[2]:
        return False
    if not timestep.is_cuda or timestep.dtype not in (torch.bfloat16, torch.float32) or len(ts_shape) < 2:
        return False
    if ts_shape[0] != shape[0] or ts_shape[1] != shape[1]:
        return False
    return timestep.numel() == shape[0] * shape[1] * table_shape[0] * shape[2]


def _can_use_fused_fp8_quantize(x: torch.Tensor, input_scale: torch.Tensor) -> bool:
    """:1021-1022 (bf16 or fp16 x). The HIP kernel also needs x 16-byte
    aligned and a float32 scale on x's device."""
    return (
        x.is_cuda
        and x.is_contiguous()
        and input_scale.numel() == 1
        and x.dtype in (torch.bfloat16, torch.float16)
        and _aligned(x)
        and input_scale.is_cuda
        and input_scale.device == x.device
        and input_scale.dtype == torch.float32
    )


def _can_use_fused_bias_add(x: torch.Tensor, bias: torch.Tensor) -> bool:
    """:1025-1034"""
    if not x.is_cuda or not x.is_contiguous() or x.dtype != torch.bfloat16:
        return False
    if x.ndim < 2 or bias.ndim != 1 or bias.shape[0] != x.shape[-1]:
        return False
    if not bias.is_cuda or bias.dtype not in (torch.bfloat16, torch.float32):
        return False
    return True


def _can_use_fused_fp8_quantize_per_head_4d(x: torch.Tensor) -> bool:
    """:1489-1499 (bf16 or fp16 x), plus the HIP kernel's layout needs (H*D in
    {1024, 2048, 4096}, x 16-byte aligned)."""
    if not x.is_cuda or not x.is_contiguous() or x.dtype not in (torch.bfloat16, torch.float16):
        return False
    if not _aligned(x):
        return False
    if x.ndim != 4:
        return False
    batch, tokens, heads, head_dim = x.shape
    if batch < 1 or tokens < 1 or heads < 1 or head_dim not in (64, 128):
        return False
    return heads * head_dim in (1024, 2048, 4096) and batch <= 65535


def _fused_video_qk_rmsnorm_rope_guard_reason(q, k, q_weight, k_weight, cos, sin) -> str | None:
    """:1513-1537, plus weight/cos dtype and device conditions of the HIP kernel."""
    if not q.is_cuda or not k.is_cuda or q.dtype != torch.bfloat16 or k.dtype != torch.bfloat16:
        return "qk_device_or_dtype"
    if q.shape != k.shape or q.ndim != 3 or q.shape[0] != 1 or q.shape[-1] != 4096:
        return "qk_shape"
    if q.shape[1] < 1:
        return "empty_tokens"
    if not q.is_contiguous() or not k.is_contiguous():
        return "qk_noncontiguous"
    if q_weight.shape != (4096,) or k_weight.shape != (4096,):
        return "qk_weight_shape"
    if cos.ndim != 4 or sin.ndim != 4 or cos.shape != sin.shape:
        return "rope_shape"
    if cos.shape[0] not in (1, q.shape[0]) or cos.shape[1] != 32 or cos.shape[2] != q.shape[1] or cos.shape[3] != 64:
        return "rope_shape"
    if not (q_weight.is_cuda and k_weight.is_cuda and cos.is_cuda and sin.is_cuda):
        return "weight_or_rope_device"
    if q_weight.dtype != k_weight.dtype or q_weight.dtype not in (torch.bfloat16, torch.float32):
        return "weight_dtype"
    if cos.dtype != sin.dtype or cos.dtype not in (torch.bfloat16, torch.float32):
        return "rope_dtype"
    if not _aligned(q) or not _aligned(k):
        return "qk_alignment"
    if not _vec_ok(q_weight, q_weight.dtype) or not _vec_ok(k_weight, q_weight.dtype):
        return "weight_alignment"
    return None


def _vec_ok(t: torch.Tensor, dtype: torch.dtype) -> bool:
    """A parameter vector the HIP kernels read 8 elements at a time, as the
    wrapper passes it (`t.to(dtype).contiguous()`): a copy is aligned; the
    tensor itself must start on an 8-element boundary."""
    if t.dtype != dtype or not t.is_contiguous():
        return True
    return _aligned(t, 8 * t.element_size())


def _can_use_fused_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, cos, sin) -> bool:
    return _fused_video_qk_rmsnorm_rope_guard_reason(q, k, q_weight, k_weight, cos, sin) is None


def _fused_video_qkv_rmsnorm_rope_pack_guard_reason(q, k, v, q_weight, k_weight, cos, sin) -> str | None:
    """:1553-1575"""
    reason = _fused_video_qk_rmsnorm_rope_guard_reason(q, k, q_weight, k_weight, cos, sin)
    if reason is not None:
        return reason
    if v.shape != q.shape:
        return "v_shape"
    if not v.is_cuda:
        return "v_device"
    if not v.is_contiguous():
        return "v_noncontiguous"
    if v.dtype != q.dtype:
        return "v_dtype"
    if not _aligned(v):
        return "v_alignment"
    return None


def _can_use_fused_video_qk_bias_rmsnorm_rope(q, k, q_bias, k_bias, q_weight, k_weight, cos, sin) -> bool:
    """:1578-1593"""
    if not _can_use_fused_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, cos, sin):
        return False
    if q_bias.shape != (4096,) or k_bias.shape != (4096,):
        return False
    if not q_bias.is_cuda or not k_bias.is_cuda:
        return False
    if q_bias.dtype not in (torch.bfloat16, torch.float32) or k_bias.dtype != q_bias.dtype:
        return False
    return _vec_ok(q_bias, q_bias.dtype) and _vec_ok(k_bias, q_bias.dtype)


def _can_use_fused_residual_gate(x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor) -> bool:
    """:1596-1609, plus the HIP kernel's needs: x and y 16-byte aligned, at
    most 65535 batches."""
    if not x.is_cuda or not y.is_cuda or x.dtype != torch.bfloat16 or y.dtype != torch.bfloat16:
        return False
    if x.shape != y.shape or x.ndim < 2 or x.shape[-1] not in (2048, 4096):
        return False
    if not x.is_contiguous() or not y.is_contiguous():
        return False
    if not _aligned(x) or not _aligned(y) or (x.ndim == 3 and x.shape[0] > 65535):
        return False
    if not gate.is_cuda or gate.dtype != torch.bfloat16:
        return False
    if gate.shape[-1] != x.shape[-1] or gate.numel() % x.shape[-1] != 0:
        return False
    return True


def _can_use_fused_head_gate_mul(out: torch.Tensor, gates: torch.Tensor, heads: int, dim_head: int) -> bool:
    """:1612-1623"""
    if not out.is_cuda or out.dtype != torch.bfloat16 or not out.is_contiguous():
        return False
    if out.ndim != 3 or heads < 1 or dim_head < 1 or out.shape[-1] != heads * dim_head:
        return False
    if not gates.is_cuda or gates.dtype != torch.bfloat16:
        return False
    if gates.shape != (out.shape[0], out.shape[1], heads):
        return False
    return True


def _can_use_fused_adazero(x: torch.Tensor, scale: torch.Tensor, shift: torch.Tensor) -> bool:
    """:1626-1637, plus conditions the reference's kernel needs but does not
    check (contiguous x) and dtype/device/alignment conditions of the HIP
    kernel (x 16-byte aligned, at most 65535 batches)."""
    if not x.is_cuda or x.dtype != torch.bfloat16:
        return False
    if x.ndim < 2 or x.shape[-1] not in (2048, 4096):
        return False
    if scale.shape[-1] != x.shape[-1] or shift.shape[-1] != x.shape[-1]:
        return False
    if scale.numel() % x.shape[-1] != 0 or shift.numel() % x.shape[-1] != 0:
        return False
    if scale.numel() != shift.numel():
        return False
    if not x.is_contiguous() or x.ndim > 3:
        return False
    if not _aligned(x) or (x.ndim == 3 and x.shape[0] > 65535):
        return False
    if not scale.is_cuda or not shift.is_cuda:
        return False
    if scale.dtype not in (torch.bfloat16, torch.float32) or shift.dtype not in (torch.bfloat16, torch.float32):
        return False
    return True


# --------------------------------------------------------------------------
# shared argument preparation
# --------------------------------------------------------------------------
def _ada_args(x: torch.Tensor, table: torch.Tensor, timestep: torch.Tensor, *indices: int):
    params = table.shape[0]
    for i in indices:
        if not -params <= i < params:
            raise IndexError(f"Ada index {i} out of range for a table with {params} rows")
    ts_view = timestep.reshape(x.shape[0], timestep.shape[1], params, x.shape[-1])
    st = ts_view.stride()
    norm = [i % params for i in indices]
    return ts_view, st, norm


def _ada_rows(x: torch.Tensor, table: torch.Tensor, timestep: torch.Tensor, *indices: int):
    """_ada_args for callers that pass the view on as pointer and strides only:
    a (B, N, P*C) timestep's (B, N, P, C) view starts where it starts and
    splits its last stride, so no view is made."""
    params, c = table.shape[0], x.shape[2]
    if timestep.ndim != 3 or timestep.shape[2] != params * c:
        return _ada_args(x, table, timestep, *indices)
    norm = []
    for i in indices:
        if not -params <= i < params:
            raise IndexError(f"Ada index {i} out of range for a table with {params} rows")
        norm.append(i % params)
    s0, s1, s2 = timestep.stride()
    return timestep, (s0, s1, c * s2, s2), norm


def _as_bnc(x: torch.Tensor) -> tuple[int, int, int]:
    if x.ndim == 2:
        return 1, x.shape[0], x.shape[1]
    return x.shape[0], x.shape[1], x.shape[2]


def _view_bnc(t: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """t as broadcast against x, seen in x's (B, N, C) form."""
    if x.ndim == 2:
        return t.expand(x.shape).unsqueeze(0)
    return t.expand(x.shape)


# --------------------------------------------------------------------------
# AdaZero family
# --------------------------------------------------------------------------
def fused_adazero(x: torch.Tensor, eps: float, scale: torch.Tensor, shift: torch.Tensor) -> torch.Tensor:
    """:8-37 — y = rms_norm(x) * (1 + scale) + shift."""
    if not _can_use_fused_adazero(x, scale, shift):
        _fallback("fused_adazero", x, scale, shift)
        return torch.nn.functional.rms_norm(x, (x.shape[-1],), eps=eps) * (1 + scale) + shift
    try:
        se = _view_bnc(scale, x)
        he = _view_bnc(shift, x)
    except RuntimeError:
        _fallback("fused_adazero", x, scale, shift)
        return torch.nn.functional.rms_norm(x, (x.shape[-1],), eps=eps) * (1 + scale) + shift
    b, n, c = _as_bnc(x)
    y = torch.empty_like(x)
    _hip("fused_adazero")
    _lib.call("oga_adazero", x.data_ptr(), y.data_ptr(), b, n, c, _ptr(se), _dt(scale), se.stride(), _ptr(he),
              _dt(shift), he.stride(), float(eps), _stream(x))
    return y


def fused_adazero_from_ada(
    x: torch.Tensor,
    eps: float,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    shift_index: int,
    scale_index: int,
    counter: str = "video",
) -> torch.Tensor:
    """:40-91 — AdaZero with shift/scale taken from table row + timestep row."""
    if not _can_use_ada_from_table(x, scale_shift_table, timestep):
        _fallback("fused_adazero_from_ada", x, scale_shift_table, timestep)
        shift, scale = _torch_ada_values_from_table(
            scale_shift_table, timestep, x.shape[0], x.shape[1], x.shape[-1], shift_index, scale_index
        )
        return fused_adazero(x, eps, scale, shift)
    _increment_ada_counter(counter)
    ts_view, st, (si, ci) = _ada_rows(x, scale_shift_table, timestep, shift_index, scale_index)
    y = torch.empty_like(x)
    _hip("fused_adazero_from_ada")
    _lib.call("oga_adazero_from_ada", x.data_ptr(), y.data_ptr(), *x.shape, scale_shift_table.data_ptr(),
              _dt(scale_shift_table), *scale_shift_table.stride(), ts_view.data_ptr(), _dt(timestep), st, si, ci,
              float(eps), _stream(x))
    return y


def _ada_rows_vec8(t: torch.Tensor, offset: int, *strides_: int) -> bool:
    """16-byte row reads of an Ada source (the C library's own check): unit
    column stride, 8-element aligned base, offset and outer strides."""
    if strides_[-1] != 1:
        return False
    es = t.element_size()
    g = 8 * es
    return t.data_ptr() % g == 0 and all((v * es) % g == 0 for v in (offset, *strides_[:-1]))


def fused_adazero_from_ada_fp8(
    x: torch.Tensor,
    eps: float,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    input_scale: torch.Tensor,
    *,
    shift_index: int,
    scale_index: int,
    counter: str = "video",
) -> torch.Tensor:
    """AdaZero from the Ada table (:40-91) handed to the FP8Linear that reads
    it (:1691-1709): the e4m3 codes of `fused_fp8_quantize_e4m3` (:144-161)
    applied to `fused_adazero_from_ada`'s output, from one HIP pass that never
    writes the bf16 rows. No single counterpart in the reference."""
    ok = (_can_use_ada_from_table(x, scale_shift_table, timestep) and _can_use_fused_fp8_quantize(x, input_scale)
          and input_scale.device == x.device and scale_shift_table.device == x.device
          and timestep.device == x.device)
    if ok:
        ts_view, st, (si, ci) = _ada_args(x, scale_shift_table, timestep, shift_index, scale_index)
        tab_s = scale_shift_table.stride()
        ok = all(_ada_rows_vec8(scale_shift_table, i * tab_s[0], tab_s[1]) for i in (si, ci)) and all(
            _ada_rows_vec8(ts_view, i * ts_view.stride(2), ts_view.stride(0), ts_view.stride(1), ts_view.stride(3))
            for i in (si, ci))
    if not ok:
        _fallback("fused_adazero_from_ada_fp8", x, scale_shift_table, timestep, input_scale)
        y = fused_adazero_from_ada(x, eps, scale_shift_table, timestep, shift_index=shift_index,
                                   scale_index=scale_index, counter=counter)
        return fused_fp8_quantize_e4m3(y, input_scale)
    _increment_ada_counter(counter)
    q = torch.empty(x.shape, device=x.device, dtype=_FP8)
    _hip("fused_adazero_from_ada_fp8")
    _lib.call("oga_adazero_from_ada_fp8", x.data_ptr(), q.data_ptr(), x.shape[0], x.shape[1], x.shape[2],
              scale_shift_table.data_ptr(), _dt(scale_shift_table), tab_s[0], tab_s[1], ts_view.data_ptr(),
              _dt(timestep), st, si, ci, float(eps), _ptr(input_scale), int(input_scale.dim() == 0), _stream(x))
    return q


def fused_adaln_affine_from_ada(
    x: torch.Tensor,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    shift_index: int,
    scale_index: int,
) -> torch.Tensor:
    """:94-141 — y = x * (1 + scale) + shift with Ada shift/scale."""
    global _VIDEO_TEXT_ADALN_CALLS
    if not _can_use_ada_from_table(x, scale_shift_table, timestep):
        _fallback("fused_adaln_affine_from_ada", x, scale_shift_table, timestep)
        shift, scale = _torch_ada_values_from_table(
            scale_shift_table, timestep, x.shape[0], x.shape[1], x.shape[-1], shift_index, scale_index
        )
        return x * (1 + scale) + shift
    _VIDEO_TEXT_ADALN_CALLS += 1
    ts_view, st, (si, ci) = _ada_rows(x, scale_shift_table, timestep, shift_index, scale_index)
    y = torch.empty_like(x)
    _hip("fused_adaln_affine_from_ada")
    _lib.call("oga_adaln_affine_from_ada", x.data_ptr(), y.data_ptr(), x.shape[0], x.shape[1], x.shape[2],
              scale_shift_table.data_ptr(), _dt(scale_shift_table), scale_shift_table.stride(0),
              scale_shift_table.stride(1), ts_view.data_ptr(), _dt(timestep), st, si, ci, _stream(x))
    return y


def fused_mul_from_ada(
    x: torch.Tensor,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    gate_index: int,
) -> torch.Tensor:
    """:695-739 — y = x * gate."""
    global _VIDEO_TEXT_ADALN_CALLS
    if not _can_use_ada_from_table(x, scale_shift_table, timestep):
        _fallback("fused_mul_from_ada", x, scale_shift_table, timestep)
        (gate,) = _torch_ada_values_from_table(
            scale_shift_table, timestep, x.shape[0], x.shape[1], x.shape[-1], gate_index
        )
        return x * gate
    _VIDEO_TEXT_ADALN_CALLS += 1
    ts_view, st, (gi,) = _ada_rows(x, scale_shift_table, timestep, gate_index)
    y = torch.empty_like(x)
    _hip("fused_mul_from_ada")
    _lib.call("oga_mul_from_ada", x.data_ptr(), y.data_ptr(), *x.shape, scale_shift_table.data_ptr(),
              _dt(scale_shift_table), scale_shift_table.stride(0), scale_shift_table.stride(1), ts_view.data_ptr(),
              _dt(timestep), st, gi, _stream(x))
    return y


# --------------------------------------------------------------------------
# residual gates and bias
# --------------------------------------------------------------------------
def fused_residual_gate_from_ada(
    x: torch.Tensor,
    y: torch.Tensor,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    gate_index: int,
    count_video_ada: bool = True,
    counter: str | None = None,
) -> torch.Tensor:
    """:640-692 — out = x + y * gate (production residual rounding)."""
    if not _can_use_ada_from_table(x, scale_shift_table, timestep) or not y.is_contiguous() or y.shape != x.shape:
        _fallback("fused_residual_gate_from_ada", x, y, scale_shift_table, timestep)
        (gate,) = _torch_ada_values_from_table(
            scale_shift_table, timestep, x.shape[0], x.shape[1], x.shape[-1], gate_index
        )
        return _simple_residual_gate(x, y, gate)
    if y.dtype != torch.bfloat16 or not y.is_cuda or not _aligned(y):
        _fallback("fused_residual_gate_from_ada", x, y)
        (gate,) = _torch_ada_values_from_table(
            scale_shift_table, timestep, x.shape[0], x.shape[1], x.shape[-1], gate_index
        )
        return _simple_residual_gate(x, y, gate)
    if counter is not None:
        _increment_ada_counter(counter)
    elif count_video_ada:
        _increment_ada_counter("video")
    else:
        _increment_ada_counter("video_text")
    ts_view, st, (gi,) = _ada_rows(x, scale_shift_table, timestep, gate_index)
    out = torch.empty_like(x)
    _hip("fused_residual_gate_from_ada")
    _lib.call("oga_residual_gate_from_ada", x.data_ptr(), y.data_ptr(), out.data_ptr(), *x.shape,
              scale_shift_table.data_ptr(), _dt(scale_shift_table), scale_shift_table.stride(0),
              scale_shift_table.stride(1), ts_view.data_ptr(), _dt(timestep), st, gi, _stream(x))
    return out


def fused_residual_gate_bias_from_ada(
    x: torch.Tensor,
    y_no_bias: torch.Tensor,
    bias: torch.Tensor,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    gate_index: int,
    count_video_ada: bool = True,
) -> torch.Tensor:
    """:204-262 — out = x + (y + bias) * gate."""
    global _VIDEO_ADA_VALUES_CALLS, _VIDEO_TEXT_ADALN_CALLS
    if (
        not _can_use_ada_from_table(x, scale_shift_table, timestep)
        or not y_no_bias.is_contiguous()
        or y_no_bias.shape != x.shape
        or not _can_use_fused_bias_add(y_no_bias, bias)
        or not _aligned(y_no_bias)
        or not (not bias.is_contiguous() or _aligned(bias, 32))
    ):
        _fallback("fused_residual_gate_bias_from_ada", x, y_no_bias, bias, scale_shift_table, timestep)
        y = y_no_bias + bias.to(y_no_bias.dtype)
        return fused_residual_gate_from_ada(
            x, y, scale_shift_table, timestep, gate_index=gate_index, count_video_ada=count_video_ada
        )
    if count_video_ada:
        _VIDEO_ADA_VALUES_CALLS += 1
    else:
        _VIDEO_TEXT_ADALN_CALLS += 1
    ts_view, st, (gi,) = _ada_rows(x, scale_shift_table, timestep, gate_index)
    bias_c = bias.contiguous()
    out = torch.empty_like(x)
    _hip("fused_residual_gate_bias_from_ada")
    _lib.call("oga_residual_gate_bias_from_ada", x.data_ptr(), y_no_bias.data_ptr(), bias_c.data_ptr(), _dt(bias_c),
              out.data_ptr(), *x.shape, scale_shift_table.data_ptr(), _dt(scale_shift_table),
              *scale_shift_table.stride(), ts_view.data_ptr(), _dt(timestep), st, gi, _stream(x))
    return out


def fused_residual_gate_adazero_from_ada(
    x: torch.Tensor,
    y: torch.Tensor,
    scale_shift_table: torch.Tensor,
    timestep: torch.Tensor,
    *,
    gate_index: int,
    shift_index: int,
    scale_index: int,
    eps: float,
    bias: torch.Tensor | None = None,
    input_scale: torch.Tensor | None = None,
    count_video_ada: bool = True,
) -> tuple[torch.Tensor, torch.Tensor]:
    """A residual gate and the AdaZero pass that reads its output, as the
    block runs them back to back (the self-attention's residual :3057-3064,
    then the cross-attention's rms_norm + AdaLN :2856-2862; the
    cross-attention's residual :2881-2888, then the feed-forward's AdaZero
    :3226-3233), in one HIP pass over the rows. Returns (x_new, out):
    x_new = `fused_residual_gate_bias_from_ada(x, y, bias, ...)` (:204-262;
    bias None: `fused_residual_gate_from_ada`, :640-692) and
    out = `fused_adazero_from_ada(x_new, eps, ...)` (:40-91), or with
    input_scale the e4m3 codes of `fused_adazero_from_ada_fp8`; both are
    bit-identical to those calls, which also serve every input the pass
    does not take (hidden size other than 4096, per-token timesteps,
    misaligned rows). No single counterpart in the reference. The Ada
    counters move as the separate calls move them."""
    global _VIDEO_ADA_VALUES_CALLS, _VIDEO_TEXT_ADALN_CALLS
    ok = (_can_use_ada_from_table(x, scale_shift_table, timestep) and x.shape[-1] == 4096
          and y.is_cuda and y.dtype == torch.bfloat16 and y.is_contiguous() and y.shape == x.shape and _aligned(y)
          and scale_shift_table.device == x.device and timestep.device == x.device and y.device == x.device)
    if ok and bias is not None:
        ok = (_can_use_fused_bias_add(y, bias) and bias.ndim == 1 and bias.dtype in (torch.bfloat16, torch.float32)
              and bias.device == x.device and (not bias.is_contiguous() or _aligned(bias, 32)))
    if ok and input_scale is not None:
        ok = _can_use_fused_fp8_quantize(x, input_scale) and input_scale.device == x.device
    if ok:
        ts_view, st, (gi, si, ci) = _ada_args(x, scale_shift_table, timestep, gate_index, shift_index, scale_index)
        tab_s = scale_shift_table.stride()
        ok = ts_view.stride(1) == 0 and all(
            _ada_rows_vec8(scale_shift_table, i * tab_s[0], tab_s[1])
            and _ada_rows_vec8(ts_view, i * ts_view.stride(2), ts_view.stride(0), ts_view.stride(1),
                               ts_view.stride(3))
            for i in (gi, si, ci))
    if not ok:
        _fallback("fused_residual_gate_adazero_from_ada", x, y, scale_shift_table, timestep)
        if bias is not None:
            x_new = fused_residual_gate_bias_from_ada(x, y, bias, scale_shift_table, timestep, gate_index=gate_index,
                                                      count_video_ada=count_video_ada)
        else:
            x_new = fused_residual_gate_from_ada(x, y, scale_shift_table, timestep, gate_index=gate_index,
                                                 count_video_ada=count_video_ada)
        if input_scale is not None:
            out = fused_adazero_from_ada_fp8(x_new, eps, scale_shift_table, timestep, input_scale,
                                             shift_index=shift_index, scale_index=scale_index)
        else:
            out = fused_adazero_from_ada(x_new, eps, scale_shift_table, timestep, shift_index=shift_index,
                                         scale_index=scale_index)
        return x_new, out
    if count_video_ada:
        _VIDEO_ADA_VALUES_CALLS += 1
    else:
        _VIDEO_TEXT_ADALN_CALLS += 1
    _increment_ada_counter("video")
    bias_c = bias.contiguous() if bias is not None else None
    x_new = torch.empty_like(x)
    out = torch.empty(x.shape, device=x.device, dtype=_FP8) if input_scale is not None else torch.empty_like(x)
    _hip("fused_residual_gate_adazero_from_ada")
    _lib.call("oga_residual_gate_adazero_from_ada", x.data_ptr(), y.data_ptr(), _ptr(bias_c),
              _dt(bias_c) if bias_c is not None else 0, _ptr(x_new), out.data_ptr(), x.shape[0], x.shape[1], x.shape[2],
              scale_shift_table.data_ptr(), _dt(scale_shift_table), tab_s[0], tab_s[1], ts_view.data_ptr(),
              _dt(timestep), st, gi, si, ci, float(eps), _ptr(input_scale),
              int(input_scale.dim() == 0) if input_scale is not None else 0, _stream(x))
    return x_new, out


def fused_residual_gate_bf16(x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """:590-611 — out = x + y * gate with gate broadcast over rows."""
    if not _can_use_fused_residual_gate(x, y, gate) or x.ndim > 3:
        _fallback("fused_residual_gate_bf16", x, y, gate)
        return x + y * gate
    try:
        ge = _view_bnc(gate, x)
    except RuntimeError:
        _fallback("fused_residual_gate_bf16", x, y, gate)
        return x + y * gate
    b, n, c = _as_bnc(x)
    out = torch.empty_like(x)
    _hip("fused_residual_gate_bf16")
    _lib.call("oga_residual_gate_bf16", x.data_ptr(), y.data_ptr(), ge.data_ptr(), ge.stride(), out.data_ptr(), b, n, c,
              _stream(x))
    return out


def fused_bias_add_bf16(x: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """:185-201 — out = x + bias.to(bf16)."""
    if not _can_use_fused_bias_add(x, bias):
        _fallback("fused_bias_add_bf16", x, bias)
        return x + bias.to(x.dtype)
    bias_c = bias.contiguous()
    out = torch.empty_like(x)
    _hip("fused_bias_add_bf16")
    _lib.call("oga_bias_add_bf16", x.data_ptr(), _ptr(bias_c), _dt(bias_c), out.data_ptr(), x.numel() // x.shape[-1],
              x.shape[-1], _stream(x))
    return out


def fused_head_gate_mul_bf16(out: torch.Tensor, gates: torch.Tensor, heads: int, dim_head: int) -> torch.Tensor:
    """:614-637 — y[b, t, h*D + d] = out[...] * gates[b, t, h]."""
    if not _can_use_fused_head_gate_mul(out, gates, heads, dim_head):
        _fallback("fused_head_gate_mul_bf16", out, gates)
        batch, tokens, _ = out.shape
        return (out.view(batch, tokens, heads, dim_head) * gates.unsqueeze(-1)).view(batch, tokens, heads * dim_head)
    y = torch.empty_like(out)
    g2 = gates.reshape(-1, heads)
    _hip("fused_head_gate_mul_bf16")
    _lib.call("oga_head_gate_mul_bf16", out.data_ptr(), _ptr(g2), g2.stride(0), g2.stride(1), y.data_ptr(),
              out.numel() // out.shape[-1], heads, dim_head, _stream(out))
    return y


# --------------------------------------------------------------------------
# FP8 quantizers
# --------------------------------------------------------------------------
def fused_fp8_quantize_e4m3(x: torch.Tensor, input_scale: torch.Tensor) -> torch.Tensor:
    """:144-161 — clamp(x * input_scale.reciprocal(), +-448).to(float8_e4m3fn)."""
    if not _can_use_fused_fp8_quantize(x, input_scale):
        _fallback("fused_fp8_quantize_e4m3", x, input_scale)
        fp8_min = torch.finfo(_FP8).min
        fp8_max = torch.finfo(_FP8).max
        return torch.clamp(x * input_scale.reciprocal(), fp8_min, fp8_max).to(_FP8)
    q = torch.empty_strided(x.shape, x.stride(), device=x.device, dtype=_FP8)
    _hip("fused_fp8_quantize_e4m3")
    _lib.call("oga_fp8_quantize_e4m3", x.data_ptr(), _xdt(x), input_scale.data_ptr(), int(input_scale.dim() == 0),
              q.data_ptr(),
              x.numel(), _stream(x))
    return q


def fused_gelu_tanh_fp8_quantize_e4m3(x: torch.Tensor, input_scale: torch.Tensor) -> torch.Tensor:
    """:164-182 — quantize gelu(x, approximate='tanh').

    The HIP path looks R(gelu(x)) up in a table of all 65536 bf16 inputs,
    built on the device with the float32 steps of torch's GPU kernel (the
    device tanhf), so the codes equal torch's."""
    if not _can_use_fused_fp8_quantize(x, input_scale):
        _fallback("fused_gelu_tanh_fp8_quantize_e4m3", x, input_scale)
        gelu = torch.nn.functional.gelu(x, approximate="tanh")
        fp8_min = torch.finfo(_FP8).min
        fp8_max = torch.finfo(_FP8).max
        return torch.clamp(gelu * input_scale.reciprocal(), fp8_min, fp8_max).to(_FP8)
    q = torch.empty_strided(x.shape, x.stride(), device=x.device, dtype=_FP8)
    _hip("fused_gelu_tanh_fp8_quantize_e4m3")
    _lib.call("oga_gelu_tanh_fp8_quantize_e4m3", x.data_ptr(), _xdt(x), input_scale.data_ptr(),
              int(input_scale.dim() == 0), q.data_ptr(),
              x.numel(), _stream(x))
    return q


def fused_fp8_quantize_e4m3_per_head_4d(
    x: torch.Tensor,
    *,
    reduce_block: int = 1024,
    quant_block: int = 1024,
) -> tuple[torch.Tensor, torch.Tensor]:
    """:265-317 — one e4m3 scale per (batch, head) of x [B, N, H, D].

    reduce_block/quant_block are accepted for signature compatibility; the HIP
    kernels tile by token rows instead."""
    del reduce_block, quant_block
    if not _can_use_fused_fp8_quantize_per_head_4d(x):
        _fallback("fused_fp8_quantize_e4m3_per_head_4d", x)
        return _torch_fp8_quantize_e4m3_per_head_4d(x)
    batch, tokens, heads, head_dim = x.shape
    lib = _lib.load()
    ws_bytes = int(lib.oga_fp8_per_head_workspace_bytes(batch, tokens, heads, head_dim))
    workspace = torch.empty((max(ws_bytes, 4) + 3) // 4, device=x.device, dtype=torch.float32)
    scale = torch.empty((batch, heads), device=x.device, dtype=torch.float32)
    q = torch.empty_strided(x.shape, x.stride(), device=x.device, dtype=_FP8)
    _hip("fused_fp8_quantize_e4m3_per_head_4d")
    _lib.call("oga_fp8_quantize_per_head", x.data_ptr(), _xdt(x), q.data_ptr(), scale.data_ptr(),
              workspace.data_ptr(), batch, tokens, heads,
              head_dim, _stream(x))
    return q, scale


# --------------------------------------------------------------------------
# Video Q/K preattention
# --------------------------------------------------------------------------
def _rope_strides(cos: torch.Tensor, batch: int):
    """cos/sin with a unit last stride; a size-1 batch dim broadcasts."""
    if cos.stride(3) != 1:
        cos = cos.contiguous()
    st = list(cos.stride())
    if cos.shape[0] == 1:
        st[0] = 0
    return cos, tuple(st)


def fused_video_qk_rmsnorm_rope(
    q: torch.Tensor,
    k: torch.Tensor,
    q_weight: torch.Tensor,
    k_weight: torch.Tensor,
    eps: float,
    cos: torch.Tensor,
    sin: torch.Tensor,
) -> tuple[torch.Tensor, torch.Tensor]:
    """:320-378 — q/k RMSNorm (full hidden size, learned weight) + split RoPE.

    Contract: q/k are [1, Nv, 4096] bf16, cos/sin are [B, 32, Nv, 64]."""
    if not _can_use_fused_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, cos, sin):
        _fallback("fused_video_qk_rmsnorm_rope", q, k, cos)
        return _torch_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, eps, cos, sin)
    qw, kw = q_weight.contiguous(), k_weight.to(q_weight.dtype).contiguous()
    cos, cst = _rope_strides(cos, q.shape[0])
    sin, sst = _rope_strides(sin, q.shape[0])
    q_out = torch.empty_like(q)
    k_out = torch.empty_like(k)
    _hip("fused_video_qk_rmsnorm_rope")
    _lib.call("oga_video_qk_rmsnorm_rope", q.data_ptr(), k.data_ptr(), qw.data_ptr(), kw.data_ptr(), _dt(qw),
              cos.data_ptr(), sin.data_ptr(),
              _dt(cos), cst, sst, q_out.data_ptr(), k_out.data_ptr(), q.shape[0], q.shape[1], q.shape[2], cos.shape[1],
              float(eps), _stream(q))
    return q_out, k_out


def fused_video_qk_rmsnorm_rope_separate(q, k, q_weight, k_weight, eps, cos, sin):
    """:432-505 — the two-launch form (one launch per tensor)."""
    if not _can_use_fused_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, cos, sin):
        _fallback("fused_video_qk_rmsnorm_rope_separate", q, k, cos)
        return _torch_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, eps, cos, sin)
    qw, kw = q_weight.contiguous(), k_weight.to(q_weight.dtype).contiguous()
    cos, cst = _rope_strides(cos, q.shape[0])
    sin, sst = _rope_strides(sin, q.shape[0])
    q_out = torch.empty_like(q)
    k_out = torch.empty_like(k)
    _hip("fused_video_qk_rmsnorm_rope_separate")
    for x, w, o in ((q, qw, q_out), (k, kw, k_out)):
        _lib.call("oga_video_rmsnorm_rope", x.data_ptr(), w.data_ptr(), _dt(w), cos.data_ptr(), sin.data_ptr(), _dt(cos),
                  cst, sst, o.data_ptr(), x.shape[0], x.shape[1], x.shape[2], cos.shape[1], float(eps), _stream(q))
    return q_out, k_out


def fused_video_qk_bias_rmsnorm_rope(q, k, q_bias, k_bias, q_weight, k_weight, eps, cos, sin):
    """:508-587 — q + q_bias and k + k_bias (bf16) before the preattention."""
    if not _can_use_fused_video_qk_bias_rmsnorm_rope(q, k, q_bias, k_bias, q_weight, k_weight, cos, sin):
        _fallback("fused_video_qk_bias_rmsnorm_rope", q, k, cos)
        q = q + q_bias.to(q.dtype)
        k = k + k_bias.to(k.dtype)
        return _torch_video_qk_rmsnorm_rope(q, k, q_weight, k_weight, eps, cos, sin)
    qw, kw = q_weight.contiguous(), k_weight.to(q_weight.dtype).contiguous()
    qb, kb = q_bias.contiguous(), k_bias.contiguous()
    cos, cst = _rope_strides(cos, q.shape[0])
    sin, sst = _rope_strides(sin, q.shape[0])
    q_out = torch.empty_like(q)
    k_out = torch.empty_like(k)
    _hip("fused_video_qk_bias_rmsnorm_rope")
    _lib.call("oga_video_qk_bias_rmsnorm_rope", q.data_ptr(), k.data_ptr(), _ptr(qb), _ptr(kb), _dt(qb), qw.data_ptr(),
              kw.data_ptr(), _dt(qw), cos.data_ptr(), sin.data_ptr(), _dt(cos), cst, sst, q_out.data_ptr(),
              k_out.data_ptr(), q.shape[0], q.shape[1],
              q.shape[2], cos.shape[1], float(eps), _stream(q))
    return q_out, k_out


def qk_rmsnorm(x: torch.Tensor, weight: torch.Tensor | None, eps: float) -> torch.Tensor:
    """The attention module's q/k RMSNorm where no RoPE follows (the text
    cross-attention, pe = None: `attn_module.q_norm(q)` / `k_norm(k)`,
    :1866-1867): torch.nn.functional.rms_norm over the last dimension. Runs
    the RMSNorm pass of the preattention kernel without its rotation for bf16
    x with 2048 or 4096 columns, otherwise the torch expression. The kernel
    takes the mean square from the exact sum of squares and rounds x * inv * w
    once, which torch's CPU rms_norm matches; torch's GPU rms_norm sums the
    squares in another float32 order and differs from it by at most one bf16
    step in rare elements, so this is not bit-identical to the GPU torch call
    it replaces (the fusion is opt-in: the block harness's `fuse_norm`)."""
    cols = x.shape[-1] if x.dim() else 0
    w = None if weight is None else weight.contiguous()
    ok = (x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous() and cols in (2048, 4096)
          and x.data_ptr() % 16 == 0
          and (w is None or (w.shape == (cols,) and w.device == x.device
                             and w.dtype in (torch.bfloat16, torch.float32)
                             and w.data_ptr() % (8 * w.element_size()) == 0)))
    if not ok:
        _fallback("qk_rmsnorm", x)
        return torch.nn.functional.rms_norm(x, (cols,), weight=weight, eps=eps)
    out = torch.empty_like(x)
    _hip("qk_rmsnorm")
    _lib.call("oga_rmsnorm", x.data_ptr(), _ptr(w), _dt(w) if w is not None else _lib.DT_BF16, out.data_ptr(),
              x.numel() // cols, cols, float(eps), _stream(x))
    return out


def fused_video_qkv_rmsnorm_rope_pack(q, k, v, q_weight, k_weight, eps, cos, sin) -> torch.Tensor | None:
    """:381-429 — packed [B, N, 3, H, D] = (rope(q), rope(k), v); None if the
    guard fails (the reference has no torch path for this op)."""
    if _fused_video_qkv_rmsnorm_rope_pack_guard_reason(q, k, v, q_weight, k_weight, cos, sin) is not None:
        _fallback("fused_video_qkv_rmsnorm_rope_pack", q, k, v, cos)
        return None
    batch, tokens, cols = q.shape
    heads = cos.shape[1]
    qw, kw = q_weight.contiguous(), k_weight.to(q_weight.dtype).contiguous()
    cos, cst = _rope_strides(cos, batch)
    sin, sst = _rope_strides(sin, batch)
    qkv = torch.empty((batch, tokens, 3, heads, cols // heads), device=q.device, dtype=q.dtype)
    _hip("fused_video_qkv_rmsnorm_rope_pack")
    _lib.call("oga_video_qkv_rmsnorm_rope_pack", q.data_ptr(), k.data_ptr(), v.data_ptr(), qw.data_ptr(),
              kw.data_ptr(), _dt(qw), cos.data_ptr(), sin.data_ptr(), _dt(cos), cst, sst, _ptr(qkv), batch,
              tokens, cols, heads, float(eps), _stream(q))
    return qkv


# --------------------------------------------------------------------------
# FP8 linear
# --------------------------------------------------------------------------
def _can_use_fp8_gemm(qflat: torch.Tensor, weight: torch.Tensor, scale_a, scale_b, bias, out_dtype) -> bool:
    """The HIP FP8 GEMM: e4m3 operands on the GPU (K a multiple of 128,
    16-byte rows), one float32 scale each, a bf16/fp16/f32 bias, bf16 or
    fp16 output."""
    if out_dtype not in (torch.bfloat16, torch.float16):
        return False
    if not (qflat.is_cuda and weight.is_cuda) or qflat.dtype != _FP8 or weight.dtype != _FP8:
        return False
    q_shape, w_shape = qflat.shape, weight.shape
    if len(q_shape) != 2 or len(w_shape) != 2 or q_shape[1] != w_shape[1]:
        return False
    q_stride, w_stride = qflat.stride(), weight.stride()
    if q_stride[1] != 1 or w_stride[1] != 1 or q_shape[1] % 128 != 0:
        return False
    if q_stride[0] % 16 or w_stride[0] % 16 or qflat.data_ptr() % 16 or weight.data_ptr() % 16:
        return False
    if w_shape[0] % 8:  # 16-byte output rows
        return False
    for s in (scale_a, scale_b):
        if not isinstance(s, torch.Tensor) or s.numel() != 1 or not s.is_cuda or s.dtype != torch.float32:
            return False
    if bias is not None:
        if not bias.is_cuda or bias.ndim != 1 or bias.shape[0] != w_shape[0]:
            return False
        if bias.dtype not in (torch.bfloat16, torch.float32, torch.float16):
            return False
    return True


def fp8_scaled_mm(
    qinput: torch.Tensor,
    weight: torch.Tensor,
    scale_a: torch.Tensor,
    scale_b: torch.Tensor,
    bias: torch.Tensor | None = None,
    *,
    out_dtype: torch.dtype = torch.bfloat16,
) -> torch.Tensor:
    """`torch._scaled_mm(qinput, weight.t(), scale_a, scale_b, out_dtype)`
    followed, if bias is given, by `out + bias.to(out.dtype)` (two roundings),
    as the reference's FP8Linear path computes (:742-759, :1691-1709).
    qinput [M, K] and weight [N, K] are float8_e4m3fn; out_dtype bf16 or
    fp16 (an fp16 model's FP8Linear) on the HIP path."""
    if not _can_use_fp8_gemm(qinput, weight, scale_a, scale_b, bias, out_dtype):
        _fallback("fp8_scaled_mm", qinput, weight)
        out = torch._scaled_mm(qinput, weight.t(), scale_a=scale_a, scale_b=scale_b, out_dtype=out_dtype,
                               use_fast_accum=True)
        if bias is not None:
            out = out + bias.to(out.dtype)
        return out
    m, k = qinput.shape
    n = weight.shape[0]
    out = torch.empty((m, n), device=qinput.device, dtype=out_dtype)
    if bias is not None and out_dtype == torch.float16:
        bias = bias.to(torch.float16)  # the reference's bias.to(out.dtype): R(bias) in fp16
    elif bias is not None and bias.dtype == torch.float16:
        bias = bias.float()  # exact; the bf16 kernel rounds it to bf16 itself
    bias_c = bias.contiguous() if bias is not None else None
    _hip("fp8_scaled_mm")
    # Split-K workspace for a last round of tiles that would not fill the
    # CUs (torch's caching allocator makes the per-call tensor cheap).
    ws_bytes = _lib.function("oga_fp8_linear_workspace_bytes")(m, n, k)
    ws = torch.empty((ws_bytes // 4,), device=qinput.device, dtype=torch.float32) if ws_bytes else None
    _lib.call("oga_fp8_linear_dt_ws", qinput.data_ptr(), qinput.stride(0), weight.data_ptr(), weight.stride(0),
              scale_a.data_ptr(), scale_b.data_ptr(), _ptr(bias_c), _any_dt(bias_c) if bias_c is not None else 0,
              out.data_ptr(), _xdt(out), n, m, n, k, _ptr(ws), ws_bytes, _stream(qinput))
    return out


def _restore_shape(output: torch.Tensor, origin_shape) -> torch.Tensor:
    if output.dim() != len(origin_shape):
        shape = list(origin_shape)
        shape[-1] = output.shape[-1]
        output = output.reshape(shape)
    return output


def fp8_linear_from_quantized_e4m3(linear: torch.nn.Module, qinput: torch.Tensor, *,
                                   out_dtype: torch.dtype) -> torch.Tensor:
    """:742-759 — FP8 GEMM on an already-quantized input, then `+ bias`."""
    origin_shape = qinput.shape
    qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
    output = fp8_scaled_mm(qflat, linear.weight, linear.input_scale, linear.weight_scale, linear.bias,
                           out_dtype=out_dtype)
    return _restore_shape(output, origin_shape)


def _can_use_fp8_linear_without_bias(linear: torch.nn.Module, x: torch.Tensor) -> bool:
    """:1037-1054 with FP8Linear recognised by its attributes (ltx_core is
    not a dependency): an e4m3 weight, input_scale, weight_scale and a bias."""
    w = getattr(linear, "weight", None)
    if not isinstance(w, torch.Tensor) or w.dtype != _FP8:
        return False
    if getattr(linear, "input_scale", None) is None or getattr(linear, "weight_scale", None) is None:
        return False
    if getattr(linear, "bias", None) is None:
        return False
    if not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float16):
        return False
    return x.shape[-1] == w.shape[1]


def fp8_linear_without_bias(linear: torch.nn.Module, x: torch.Tensor, *,
                            out_dtype: torch.dtype) -> torch.Tensor | None:
    """:762-781 — quantize + FP8 GEMM, bias left to the caller; None if the
    module is not an FP8 linear."""
    if not _can_use_fp8_linear_without_bias(linear, x):
        return None
    origin_shape = x.shape
    qinput = fused_fp8_quantize_e4m3(x.contiguous(), linear.input_scale)
    qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
    output = fp8_scaled_mm(qflat, linear.weight, linear.input_scale, linear.weight_scale, None, out_dtype=out_dtype)
    return _restore_shape(output, origin_shape)


def fp8_linear_forward(linear: torch.nn.Module, x: torch.Tensor) -> torch.Tensor:
    """The patched `FP8Linear.forward` of `patch_ltx_fp8_quantize(triton_bias_add=True)`
    (:1671-1718): quantize x with the module's input_scale, FP8 GEMM to
    x.dtype (bf16 or fp16), then the exact bias add in that dtype — here
    fused into the GEMM epilogue."""
    origin_shape = x.shape
    qinput = fused_fp8_quantize_e4m3(x.contiguous(), linear.input_scale)
    qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
    output = fp8_scaled_mm(qflat, linear.weight, linear.input_scale, linear.weight_scale,
                           getattr(linear, "bias", None), out_dtype=x.dtype)
    return _restore_shape(output, origin_shape)


# --------------------------------------------------------------------------
# Q/K/V projections of video self-attention
# --------------------------------------------------------------------------
def _is_fp8_linear(linear) -> bool:
    """FP8Linear recognised by its attributes (ltx_core is not a dependency)."""
    w = getattr(linear, "weight", None)
    return (isinstance(w, torch.Tensor) and w.dtype == _FP8 and getattr(linear, "input_scale", None) is not None
            and getattr(linear, "weight_scale", None) is not None)


_EQUAL_MEMO: dict = {}
_FROZEN_SCALES = False


def set_frozen_fp8_scales(frozen: bool) -> bool:
    """Declares whether the FP8 linears' scale tensors stay fixed while the
    flag is on (a loaded model's do). On: the Q/K/V guards remember the
    result of comparing a tuple of scale tensors, which saves a
    device-to-host synchronisation per call (each torch.equal on GPU tensors
    is one, and it drains the launch queue in the middle of a block). The
    remembered result is used only while every tensor is the same object,
    with the same storage and, where torch tracks one, the same in-place
    version counter; writes that bypass the counter (through `.data`, or
    to an inference tensor inside inference mode) are not seen, which is
    what the caller promises not to make. Off (the default): every call
    compares, as the reference does (:1209-1214, :1258-1259). Returns the
    previous setting."""
    global _FROZEN_SCALES
    prev = _FROZEN_SCALES
    _FROZEN_SCALES = bool(frozen)
    if not _FROZEN_SCALES:
        _EQUAL_MEMO.clear()
    return prev


class frozen_fp8_scales:
    """`with frozen_fp8_scales(): ...` turns set_frozen_fp8_scales on for the
    block and restores the previous setting after it."""

    def __enter__(self):
        self._prev = set_frozen_fp8_scales(True)
        return self

    def __exit__(self, *exc):
        set_frozen_fp8_scales(self._prev)
        return False


def _version_or_none(t: torch.Tensor):
    """The in-place version counter, or None for a tensor without one (an
    inference tensor: reading its `_version` raises)."""
    try:
        return t._version
    except RuntimeError:
        return None


def _all_equal(tensors) -> bool:
    """torch.equal of every tensor with the first, as the reference's guards
    evaluate it; remembered per tuple of tensors while
    set_frozen_fp8_scales is on."""
    if not _FROZEN_SCALES:
        return all(torch.equal(tensors[0], t) for t in tensors[1:])
    key = tuple(id(t) for t in tensors)
    state = tuple((t.data_ptr(), _version_or_none(t)) for t in tensors)
    memo = _EQUAL_MEMO.get(key)
    if memo is not None:
        refs, old_state, result = memo
        if old_state == state and all(r() is t for r, t in zip(refs, tensors)):
            return result
    result = all(torch.equal(tensors[0], t) for t in tensors[1:])
    if len(_EQUAL_MEMO) >= 1024:
        _EQUAL_MEMO.clear()
    _EQUAL_MEMO[key] = (tuple(weakref.ref(t) for t in tensors), state, result)
    return result


def _scale_fits(scale: torch.Tensor, length: int) -> bool:
    """`_scale_row` (:1281-1287) accepts a scalar or `length` values."""
    return scale.numel() in (1, length)


def _can_use_video_qkv_shared(attn: torch.nn.Module, x: torch.Tensor, names: tuple[str, ...],
                              grouped: bool) -> bool:
    """:1070-1096 (shared quantized input) and, with `grouped`, :1187-1233 /
    :1236-1278 (grouped scaled-mm): x (1, N, 4096) contiguous bf16/fp16; the
    linears are FP8 with a bias and one input scale; grouped also needs
    square 4096 linears and weight scales `_scale_row` accepts."""
    if not x.is_cuda or not x.is_contiguous() or x.dtype not in (torch.bfloat16, torch.float16):
        return False
    return _video_qkv_linears_ok(attn, x, names, grouped)


def _video_qkv_linears_ok(attn: torch.nn.Module, x: torch.Tensor, names: tuple[str, ...], grouped: bool) -> bool:
    """The shape and linear checks of `_can_use_video_qkv_shared` for an input
    x of any dtype (bf16 activations or their e4m3 codes)."""
    if x.ndim != 3 or x.shape[0] != 1 or x.shape[1] < 1 or x.shape[-1] != 4096:
        return False
    linears = [getattr(attn, n, None) for n in names]
    if not all(_is_fp8_linear(lin) for lin in linears):
        return False
    if not all(getattr(lin, "bias", None) is not None for lin in linears):
        return False
    s0 = linears[0].input_scale
    if not _all_equal([lin.input_scale for lin in linears]):
        return False
    if not grouped:
        return True
    if not all(tuple(lin.weight.shape) == (x.shape[-1], x.shape[-1]) for lin in linears):
        return False
    rows = x.shape[0] * x.shape[1]
    return _scale_fits(s0, rows) and all(_scale_fits(lin.weight_scale, lin.weight.shape[0]) for lin in linears)


def _grouped_hip_ok(linears, qflat: torch.Tensor, out_dtype: torch.dtype) -> bool:
    """The HIP grouped GEMM: bf16 outputs, scalar float32 scales, e4m3 weights
    with 16-byte rows, 16-byte aligned bf16 biases."""
    if out_dtype != torch.bfloat16 or not qflat.is_cuda or qflat.stride(1) != 1 or qflat.data_ptr() % 16:
        return False
    s0 = linears[0].input_scale
    if s0.numel() != 1 or s0.dtype != torch.float32 or not s0.is_cuda:
        return False
    for lin in linears:
        w, ws, b = lin.weight, lin.weight_scale, lin.bias
        if not w.is_cuda or w.stride(1) != 1 or w.stride(0) != qflat.shape[1] or w.data_ptr() % 16:
            return False
        if ws.numel() != 1 or ws.dtype != torch.float32 or not ws.is_cuda:
            return False
        if b.dtype != torch.bfloat16 or not b.is_cuda or not b.is_contiguous() or b.data_ptr() % 16:
            return False
    return True


def _grouped_launch(linears, qflat: torch.Tensor, weight_scales, outs, ldo: int) -> None:
    """One launch of the grouped FP8 GEMM: linear i's weight, `weight_scales[i]`
    and bias into `outs[i]` (column blocks with row stride `ldo`)."""
    import ctypes

    m, k = qflat.shape
    n = linears[0].weight.shape[0]
    lib = _lib.load()
    ws_bytes = int(lib.oga_fp8_linear_workspace_bytes(m, n * len(linears), k))
    ws = torch.empty((ws_bytes // 4,), device=qflat.device, dtype=torch.float32) if ws_bytes else None
    arr = ctypes.c_void_p * len(linears)
    w_p = arr(*[lin.weight.data_ptr() for lin in linears])
    s_p = arr(*[s.data_ptr() for s in weight_scales])
    b_p = arr(*[lin.bias.data_ptr() for lin in linears])
    o_p = arr(*[o.data_ptr() for o in outs])
    _hip("fp8_grouped_linear")
    _lib.call("oga_fp8_linear_grouped_ws", qflat.data_ptr(), qflat.stride(0), ctypes.addressof(w_p), k,
              linears[0].input_scale.data_ptr(), ctypes.addressof(s_p), ctypes.addressof(b_p), _lib.DT_BF16,
              ctypes.addressof(o_p), ldo, m, n, len(linears), k, _ptr(ws), ws_bytes, _stream(qflat))


def _packed_hip_ok(linears, qflat: torch.Tensor, out_dtype: torch.dtype) -> bool:
    """The grouped kernel can write the packed output: grouped-kernel operands
    and equal square weights."""
    n = linears[0].weight.shape[0]
    return _grouped_hip_ok(linears, qflat, out_dtype) and all(tuple(lin.weight.shape) == (n, qflat.shape[1])
                                                              for lin in linears)


def _fp8_grouped_linear(linears, qinput: torch.Tensor, out_dtype: torch.dtype) -> tuple[torch.Tensor, ...]:
    """One quantized input through several FP8 linears with their own weight
    scales and biases: R(R(acc * sa * sb_i) + R(bias_i)) per linear, one HIP
    launch for all; otherwise each as `fp8_linear_from_quantized_e4m3`."""
    qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
    if not _grouped_hip_ok(linears, qflat, out_dtype):
        _fallback("fp8_grouped_linear", qinput)
        return tuple(fp8_linear_from_quantized_e4m3(lin, qinput, out_dtype=out_dtype) for lin in linears)
    m = qflat.shape[0]
    n = linears[0].weight.shape[0]
    outs = [torch.empty((m, n), device=qflat.device, dtype=out_dtype) for _ in linears]
    _grouped_launch(linears, qflat, [lin.weight_scale for lin in linears], outs, n)
    if qinput.dim() == 3:
        outs = [o.reshape(qinput.shape[0], qinput.shape[1], n) for o in outs]
    return tuple(outs)


def fp8_qkv_from_shared_quantized_input(attn: torch.nn.Module, x: torch.Tensor):
    """:805-820 — Q/K/V FP8 linears from one quantized input (to_q's input
    scale, equal for all three); None when the guard fails."""
    if not _can_use_video_qkv_shared(attn, x, ("to_q", "to_k", "to_v"), grouped=False):
        return None
    qinput = fused_fp8_quantize_e4m3(x.contiguous(), attn.to_q.input_scale)
    return (fp8_linear_from_quantized_e4m3(attn.to_q, qinput, out_dtype=x.dtype),
            fp8_linear_from_quantized_e4m3(attn.to_k, qinput, out_dtype=x.dtype),
            fp8_linear_from_quantized_e4m3(attn.to_v, qinput, out_dtype=x.dtype))


# The grouped projections' bookkeeping, as the reference keeps it for
# `fp8_qkv_from_grouped_mm` / `fp8_qk_from_grouped_mm` (:1926-1937,
# :2114-2178): successful calls, fallbacks by reason (a guard's reason or an
# exception's type name) and, for the first `checks` calls after a reset,
# error statistics of the projections against the per-linear FP8 linears.
_GROUPED_STATS = {
    "qkv": {"calls": 0, "fallbacks": 0, "fallback_reasons": {}, "checks": [], "check_limit": 0},
    "qk": {"calls": 0, "fallbacks": 0, "fallback_reasons": {}, "checks": [], "check_limit": 0},
}
_GROUPED_NAMES = {"qkv": ("to_q", "to_k", "to_v"), "qk": ("to_q", "to_k")}


def _record_grouped_fallback(kind: str, reason: str) -> None:
    """:2159-2176"""
    st = _GROUPED_STATS[kind]
    st["fallbacks"] += 1
    st["fallback_reasons"][reason] = st["fallback_reasons"].get(reason, 0) + 1


def _reset_grouped_stats(kind: str, checks: int) -> None:
    st = _GROUPED_STATS[kind]
    st["calls"] = 0
    st["fallbacks"] = 0
    st["fallback_reasons"] = {}
    st["checks"] = []
    st["check_limit"] = max(0, int(checks)) * len(_GROUPED_NAMES[kind])


def reset_video_qkv_grouped_mm_stats(checks: int = 0) -> None:
    """Zeroes the grouped Q/K/V counters as patch_ltx_video_qkv_grouped_mm(checks)
    does (:2114-2123); the first `checks` calls are then compared with the
    per-linear projections and recorded."""
    _reset_grouped_stats("qkv", checks)


def reset_video_qk_grouped_mm_stats(checks: int = 0) -> None:
    """As reset_video_qkv_grouped_mm_stats for the grouped Q/K form (:2137-2146)."""
    _reset_grouped_stats("qk", checks)


def _collect_grouped(kind: str) -> dict:
    st = _GROUPED_STATS[kind]
    return {"calls": st["calls"], "fallbacks": st["fallbacks"], "fallback_reasons": dict(st["fallback_reasons"]),
            "checks": list(st["checks"])}


def collect_video_qkv_grouped_mm_stats() -> dict:
    """:2127-2133"""
    return _collect_grouped("qkv")


def collect_video_qk_grouped_mm_stats() -> dict:
    """:2150-2156"""
    return _collect_grouped("qk")


def _grouped_guard_reason(attn: torch.nn.Module, x: torch.Tensor, names: tuple[str, ...]) -> str | None:
    """:1187-1233 (Q/K/V) and :1236-1278 (Q/K), with FP8Linear recognised by
    its attributes and the same reasons as the reference records. The
    reference's first three reasons (no torch._scaled_grouped_mm, ltx_core
    import, the TRT-LLM branch) have no counterpart here: the grouped GEMM is
    this library's."""
    if not x.is_cuda or not x.is_contiguous() or x.dtype not in (torch.bfloat16, torch.float16):
        return "input"
    if x.ndim != 3 or x.shape[0] != 1 or x.shape[1] < 1 or x.shape[-1] != 4096:
        return "shape"
    linears = [getattr(attn, n, None) for n in names]
    if not all(_is_fp8_linear(lin) for lin in linears):
        return "linear_type"
    if not all(getattr(lin, "bias", None) is not None for lin in linears):
        return "bias"
    if not _all_equal([lin.input_scale for lin in linears]):
        return "input_scale"
    feats = [_features(lin) for lin in linears]
    if not all(fi == x.shape[-1] and fo == x.shape[-1] for fi, fo in feats):
        return "features"
    rows = x.shape[0] * x.shape[1]
    if not (_scale_fits(linears[0].input_scale, rows)
            and all(_scale_fits(lin.weight_scale, fo) for lin, (_, fo) in zip(linears, feats))):
        return "scale_shape"
    return None


def _record_grouped_check(kind: str, attn: torch.nn.Module, x: torch.Tensor, outs) -> None:
    """:1438-1486 — error statistics of the grouped projections against each
    linear's own FP8 forward, for the first checks after a reset."""
    st = _GROUPED_STATS[kind]
    if len(st["checks"]) >= st["check_limit"]:
        return
    with torch.no_grad():
        for name, out in zip(("q", "k", "v"), outs):
            ref = fp8_linear_forward(getattr(attn, "to_" + name), x)
            diff = (out.float() - ref.float()).abs()
            denom = ref.float().abs().clamp_min(1e-6)
            st["checks"].append({"tensor": name, "max_abs": float(diff.max().item()),
                                 "mean_abs": float(diff.mean().item()),
                                 "rms": float(torch.sqrt(torch.mean(diff.square())).item()),
                                 "mean_rel": float((diff / denom).mean().item())})


def _grouped_projections(kind: str, attn: torch.nn.Module, x: torch.Tensor):
    """The body of fp8_qkv_from_grouped_mm / fp8_qk_from_grouped_mm: guard
    (reason recorded), one quantization with to_q's input scale, one grouped
    GEMM launch; an exception is recorded by type and gives None, as the
    reference's try/except does (:919-921, :953-955). Under
    OPENGENIE_AMD_STRICT the exception propagates instead."""
    reason = _grouped_guard_reason(attn, x, _GROUPED_NAMES[kind])
    if reason is not None:
        _record_grouped_fallback(kind, reason)
        return None
    try:
        linears = tuple(getattr(attn, n) for n in _GROUPED_NAMES[kind])
        qinput = fused_fp8_quantize_e4m3(x.contiguous(), attn.to_q.input_scale)
        outs = _fp8_grouped_linear(linears, qinput, x.dtype)
        _record_grouped_check(kind, attn, x, outs)
        _GROUPED_STATS[kind]["calls"] += 1
        return outs
    except _lib.LibraryMissing:
        raise
    except Exception as exc:
        if _strict():
            raise
        _record_grouped_fallback(kind, type(exc).__name__)
        return None


def fp8_qkv_from_grouped_mm(attn: torch.nn.Module, x: torch.Tensor):
    """:890-925 — exact Q/K/V projections as one grouped FP8 GEMM with each
    linear's own weight scale and bias (one launch over the three linears'
    tiles); None when the guard fails or the launch raises (reason recorded,
    collect_video_qkv_grouped_mm_stats)."""
    return _grouped_projections("qkv", attn, x)


def fp8_qkv_from_quantized_e4m3(attn: torch.nn.Module, qinput: torch.Tensor, *, out_dtype: torch.dtype):
    """The grouped Q/K/V projection of `fp8_qkv_from_grouped_mm` (:890-925)
    on an input already quantized with to_q's input scale (as
    `fused_adazero_from_ada_fp8` leaves it); None when the guard fails."""
    if qinput.dtype != _FP8 or not qinput.is_cuda or not qinput.is_contiguous():
        return None
    if not _video_qkv_linears_ok(attn, qinput, ("to_q", "to_k", "to_v"), grouped=True):
        return None
    return _fp8_grouped_linear((attn.to_q, attn.to_k, attn.to_v), qinput, out_dtype)


def fp8_kv_from_grouped_mm(attn: torch.nn.Module, context: torch.Tensor):
    """The text cross-attention's K and V projections of the encoder states
    (the attention module's to_k / to_v FP8Linears, :1691-1709 each, inside
    the cross-attention's `attn(attn_input, context=...)`, :2880) as one
    grouped FP8 GEMM when the
    two linears share their input scale: one quantization (to_k's scale), one
    launch over both linears' tiles, each with its own weight scale and bias.
    No counterpart in the reference; the roundings are those of the two
    forwards (R(R(acc * sa * sb_i) + R(bias_i))), only the float32 sum order
    of a split tile's K-chunks may differ. None when the guard fails (the
    caller then runs the two forwards)."""
    if _grouped_guard_reason(attn, context, ("to_k", "to_v")) is not None:
        return None
    qinput = fused_fp8_quantize_e4m3(context.contiguous(), attn.to_k.input_scale)
    return _fp8_grouped_linear((attn.to_k, attn.to_v), qinput, context.dtype)


def fp8_qk_from_grouped_mm(attn: torch.nn.Module, x: torch.Tensor):
    """:927-955 — exact Q/K projections as one grouped FP8 GEMM; None when the
    guard fails or the launch raises (reason recorded,
    collect_video_qk_grouped_mm_stats)."""
    return _grouped_projections("qk", attn, x)


# --------------------------------------------------------------------------
# Packed Q/K/V projections (:822-887) and their fallback/check bookkeeping
# (:1915-1924, :2072-2110, :2179-2198)
# --------------------------------------------------------------------------
_PACKED_STATS = {
    "packed_linear": {"calls": 0, "fallbacks": 0, "fallback_reasons": {}},
    "packed_requant": {"calls": 0, "fallbacks": 0, "fallback_reasons": {}, "checks": []},
}
_PACKED_REQUANT_CHECK_LIMIT = 0


def _record_packed_fallback(kind: str, reason: str) -> None:
    st = _PACKED_STATS[kind]
    st["fallbacks"] += 1
    st["fallback_reasons"][reason] = st["fallback_reasons"].get(reason, 0) + 1


def reset_video_qkv_packed_stats(requant_checks: int = 0) -> None:
    """Zeroes the packed-projection counters (what the reference's
    patch_ltx_video_qkv_packed_linear / _requant(checks) do to them, :2072-2100);
    `requant_checks` calls of the requantized form are compared with the
    per-linear projections and recorded."""
    global _PACKED_REQUANT_CHECK_LIMIT
    for kind, st in _PACKED_STATS.items():
        st["calls"] = 0
        st["fallbacks"] = 0
        st["fallback_reasons"] = {}
        if kind == "packed_requant":
            st["checks"] = []
    _PACKED_REQUANT_CHECK_LIMIT = max(0, int(requant_checks)) * 3


def collect_video_qkv_packed_linear_stats() -> dict:
    """:2082-2087"""
    st = _PACKED_STATS["packed_linear"]
    return {"calls": st["calls"], "fallbacks": st["fallbacks"], "fallback_reasons": dict(st["fallback_reasons"])}


def collect_video_qkv_packed_requant_stats() -> dict:
    """:2104-2110"""
    st = _PACKED_STATS["packed_requant"]
    return {"calls": st["calls"], "fallbacks": st["fallbacks"], "fallback_reasons": dict(st["fallback_reasons"]),
            "checks": list(st["checks"])}


def _features(linear) -> tuple[int, int]:
    """(in_features, out_features) of an FP8 linear; from the e4m3 weight's
    [out, in] shape when the module carries no such attributes."""
    w = linear.weight
    return int(getattr(linear, "in_features", w.shape[1])), int(getattr(linear, "out_features", w.shape[0]))


def _packed_guard_reason(attn: torch.nn.Module, x: torch.Tensor, *, equal_weight_scales: bool) -> str | None:
    """:1099-1145 (equal_weight_scales) and :1146-1185, with FP8Linear
    recognised by its attributes; the same reasons as the reference records."""
    if not x.is_cuda or not x.is_contiguous() or x.dtype not in (torch.bfloat16, torch.float16):
        return "input"
    if x.ndim != 3 or x.shape[0] != 1 or x.shape[1] < 1 or x.shape[-1] != 4096:
        return "shape"
    linears = (getattr(attn, "to_q", None), getattr(attn, "to_k", None), getattr(attn, "to_v", None))
    if not all(_is_fp8_linear(lin) for lin in linears):
        return "linear_type"
    if not all(getattr(lin, "bias", None) is not None for lin in linears):
        return "bias"
    q, k, v = linears
    if not _all_equal([q.input_scale, k.input_scale, v.input_scale]):
        return "input_scale"
    if equal_weight_scales and not _all_equal([q.weight_scale, k.weight_scale, v.weight_scale]):
        return "weight_scale"
    feats = [_features(lin) for lin in linears]
    if not all(fi == x.shape[-1] and fo == x.shape[-1] for fi, fo in feats):
        return "features"
    return None


def _split_packed(output: torch.Tensor, x: torch.Tensor, out_features: int):
    """(M, 3*out) -> the reference's `output.split(out_features, dim=-1)` of
    the (B, N, 3*out) view."""
    if output.dim() != len(x.shape):
        output = output.reshape(x.shape[0], x.shape[1], output.shape[-1])
    return output.split(out_features, dim=-1)


def fp8_qkv_from_packed_linear(attn: torch.nn.Module, x: torch.Tensor):
    """:822-850 — exact Q/K/V projections as one packed FP8 matmul, for three
    FP8 linears with equal input and equal weight scales: R(R(acc * sa * sb) +
    R(bias)) over the packed [Wq; Wk; Wv], returned as the three column views
    of one (B, N, 3*4096) output. Here one launch of the grouped kernel writes
    each linear's columns into that output (no packed copy of the weights).
    None when the guard fails or the launch raises (reason recorded)."""
    reason = _packed_guard_reason(attn, x, equal_weight_scales=True)
    if reason is not None:
        _record_packed_fallback("packed_linear", reason)
        return None
    try:
        lins = (attn.to_q, attn.to_k, attn.to_v)
        qinput = fused_fp8_quantize_e4m3(x.contiguous(), attn.to_q.input_scale)
        qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
        n = _features(attn.to_q)[1]
        m, k = qflat.shape
        if _packed_hip_ok(lins, qflat, x.dtype):
            output = torch.empty((m, 3 * n), device=qflat.device, dtype=x.dtype)
            _grouped_launch(lins, qflat, [attn.to_q.weight_scale] * 3, [output[:, i * n:(i + 1) * n] for i in range(3)],
                            3 * n)
        else:
            wp = torch.cat([lin.weight for lin in lins], dim=0)
            bp = torch.cat([lin.bias for lin in lins], dim=0)
            output = fp8_scaled_mm(qflat, wp, attn.to_q.input_scale, attn.to_q.weight_scale, bp, out_dtype=x.dtype)
        _PACKED_STATS["packed_linear"]["calls"] += 1
        return _split_packed(output, x, n)
    except _lib.LibraryMissing:
        raise
    except Exception as exc:  # the reference counts the exception and returns None (:847-849)
        if _strict():
            raise
        _record_packed_fallback("packed_linear", type(exc).__name__)
        return None


def _requantized_packed(attn: torch.nn.Module) -> dict:
    """:1311-1345 — the packed weight requantized to one common scale (the
    largest of the three weight scales): e4m3(clamp(W.float() * ws / common,
    +-448)) per linear, cached on the module by weight/bias pointers and scale
    values. A one-time weight transform, evaluated with the reference's own
    torch expression on the weights' device."""
    scales = (attn.to_q.weight_scale, attn.to_k.weight_scale, attn.to_v.weight_scale)
    key = (attn.to_q.weight.data_ptr(), attn.to_k.weight.data_ptr(), attn.to_v.weight.data_ptr(),
           attn.to_q.bias.data_ptr(), attn.to_k.bias.data_ptr(), attn.to_v.bias.data_ptr(),
           tuple(float(s.detach().float().item()) for s in scales))
    cached = getattr(attn, "_oga_qkv_packed_requant_cache", None)
    if cached is not None and cached.get("key") == key:
        return cached
    common = torch.stack([s.detach().float().reshape(()) for s in scales]).amax().contiguous()

    def requant(linear):
        dequant = linear.weight.float() * linear.weight_scale.detach().float()
        return torch.clamp(dequant / common, -_FP8_MAX, _FP8_MAX).to(_FP8)

    packed = {
        "key": key,
        "weight": torch.cat((requant(attn.to_q), requant(attn.to_k), requant(attn.to_v)), dim=0).contiguous(),
        "weight_scale": common,
        "bias": torch.cat((attn.to_q.bias, attn.to_k.bias, attn.to_v.bias), dim=0).contiguous(),
    }
    attn._oga_qkv_packed_requant_cache = packed
    return packed


def _record_packed_requant_check(attn: torch.nn.Module, x: torch.Tensor, outs) -> None:
    """:1412-1440 — error statistics of the requantized projections against
    the per-linear FP8 projections, for the first checks."""
    st = _PACKED_STATS["packed_requant"]
    if len(st["checks"]) >= _PACKED_REQUANT_CHECK_LIMIT:
        return
    with torch.no_grad():
        for name, lin, out in zip(("q", "k", "v"), (attn.to_q, attn.to_k, attn.to_v), outs):
            ref = fp8_linear_forward(lin, x)
            diff = (out.float() - ref.float()).abs()
            denom = ref.float().abs().clamp_min(1e-6)
            st["checks"].append({"tensor": name, "max_abs": float(diff.max().item()),
                                 "mean_abs": float(diff.mean().item()),
                                 "rms": float(torch.sqrt(torch.mean(diff.square())).item()),
                                 "mean_rel": float((diff / denom).mean().item())})


def fp8_qkv_from_packed_requant(attn: torch.nn.Module, x: torch.Tensor):
    """:852-887 — Q/K/V as one packed FP8 matmul after requantizing the three
    weights to their largest weight scale. Not exact to the checkpoint weights
    (the reference keeps it behind --allow-quality-risk-packed-qkv-requant,
    official_ltx23_benchmark.py:539-544). One FP8 GEMM of N = 3*4096 with the
    bias epilogue; the three column views of its output. None when the guard
    fails or the launch raises (reason recorded)."""
    reason = _packed_guard_reason(attn, x, equal_weight_scales=False)
    if reason is not None:
        _record_packed_fallback("packed_requant", reason)
        return None
    try:
        packed = _requantized_packed(attn)
        qinput = fused_fp8_quantize_e4m3(x.contiguous(), attn.to_q.input_scale)
        qflat = qinput.reshape(-1, qinput.shape[-1]) if qinput.dim() == 3 else qinput
        output = fp8_scaled_mm(qflat, packed["weight"], attn.to_q.input_scale, packed["weight_scale"],
                               packed["bias"], out_dtype=x.dtype)
        q, k, v = _split_packed(output, x, _features(attn.to_q)[1])
        _record_packed_requant_check(attn, x, (q, k, v))
        _PACKED_STATS["packed_requant"]["calls"] += 1
        return q, k, v
    except _lib.LibraryMissing:
        raise
    except Exception as exc:  # :884-886
        if _strict():
            raise
        _record_packed_fallback("packed_requant", type(exc).__name__)
        return None
