"""HF transformers attention functions that run decode steps on the HIP kernels.

Reference: fskernels/triton/triton_gqa_decode_hf.py:218-258
(custom_hf_decode_attention_forward) and
fskernels/triton/triton_gqa_decode_hf_fp8.py:230-283
(custom_hf_decode_attention_forward_fp8).  They have the signature of
transformers' ``eager_attention_forward`` and are installed the way the
reference's scripts install theirs (benchmarks/run_hf_model_triton.py:9)::

    import transformers.models.qwen3.modeling_qwen3 as qwen3_mod
    qwen3_mod.eager_attention_forward = custom_hf_decode_attention_forward

or with ``patch_hf_attention()`` / ``patched_hf_attention()``.

A decode step (one query position) attends over the cache the model hands
in: key/value states [B, Hkv, S, D] from a dynamic cache (S = the sequence so
far) or a static cache (S = its capacity).  The attended range of each
sequence is computed on the device (see _decode_bounds), so the step needs no
host synchronisation and can be captured in a HIP graph.  Other calls
(prefill) go to transformers' own eager attention, as in the reference.

Differences from the reference, all deliberate:

* Decode is recognised by ``q_len == 1``.  The reference also requires
  ``past_key_values`` and ``cache_position`` in the keyword arguments; the
  installed transformers (5.x) passes neither on to the attention function,
  so that patch never takes its decode path there.  Without
  ``cache_position`` the range comes from the attention mask.
* A sliding window attends the last ``sliding_window`` positions
  ``[len - window, len)``.  The reference passes the clamped length as the end
  of the range (:244-250), which attends the wrong tokens once
  ``len > window``.
* ``scaling`` is the softmax scale the kernels use (the reference kernels use
  1/sqrt(D), the value Qwen3 passes).
* The fp8 path honours a sliding window too.
* With ``cache_position`` the mask is not read, as in the reference; without
  it, the mask's attended positions must form one contiguous range per
  sequence (true of causal, padding, static-cache and sliding-window masks).
"""
from __future__ import annotations

import contextlib
from typing import Optional, Tuple

import torch

from fasterkernels_amd import native as nat

from .decode import (_on_gpu, _stream, decode_hf, decode_quantizing_to_fp8, flash_decode_gqa_hf_dense_optimized,
                     flash_decode_gqa_hf_fp8, quantize_each_to_fp8)

_MASK_DTYPES = (torch.bool, torch.float16, torch.bfloat16, torch.float32)

try:  # captured before anything is patched, as the reference module does (:3)
    from transformers.models.qwen3.modeling_qwen3 import eager_attention_forward as _native_eager
except ImportError:  # pragma: no cover - transformers missing
    _native_eager = None

if getattr(_native_eager, "_fsk_patch", False):  # imported after a patch was installed by hand
    raise ImportError("fskernels.hip.hf must be imported before eager_attention_forward is patched")


def native_eager_attention_forward(*args, **kwargs):
    if _native_eager is None:
        raise RuntimeError("transformers is not installed")
    return _native_eager(*args, **kwargs)


def _decode_bounds(query_states: torch.Tensor, key_states: torch.Tensor, attention_mask,
                   kwargs) -> Optional[Tuple[torch.Tensor, Optional[torch.Tensor]]]:
    """(cache_lens, start_offsets) of a decode step, or None for other calls.

    All values are computed on the device, in one launch:
    * with ``cache_position`` (transformers versions that pass it, and the
      reference's contract): length cache_position[-1] + 1 and, for a sliding
      window, start max(0, length - window);
    * otherwise from the attention mask's row for the query, [B, 1, 1, S]
      (0 or True = attended): the first and one past the last attended
      position, which covers left padding, a static cache's unused tail and
      sliding windows (the attended positions must be contiguous);
    * without a mask: all S positions, and the sliding window if one is given.
    """
    bsz, _, q_len, _ = query_states.shape
    if q_len != 1:
        return None
    _on_gpu(query_states, "query_states")
    S = key_states.shape[2]
    source = _range_source(query_states, key_states, attention_mask, kwargs)
    if source is not None:
        return nat.ext().bounds(query_states, bsz, S, *source, _stream(query_states))
    cache_position = kwargs.get("cache_position")
    return _torch_bounds(bsz, S, query_states.device, attention_mask if cache_position is None else None,
                         cache_position, kwargs.get("sliding_window"))


def _range_source(query_states, key_states, attention_mask, kwargs):
    """(mask, position, window) that the kernels take the range from, or None
    where they do not read this mask or position type."""
    S = key_states.shape[2]
    position = kwargs.get("cache_position")
    if not query_states.is_cuda or not 0 < S < 1 << 31:
        return None
    if position is not None:
        attention_mask = None
        if not (position.dtype is torch.int64 and position.dim() == 1 and position.is_cuda):
            return None
    elif attention_mask is not None and not (attention_mask.dtype in _MASK_DTYPES and attention_mask.dim() == 4):
        return None
    window = kwargs.get("sliding_window")
    return attention_mask, position, None if window is None else int(window)


def _torch_bounds(bsz, S, dev, attention_mask, cache_position, window):
    """_decode_bounds in torch operations, for the mask and position types
    that the kernel does not read (integer and fp64 masks, other positions)."""
    if cache_position is not None:
        lens = (cache_position[-1:] + 1).to(torch.int32).expand(bsz).contiguous()
    elif attention_mask is not None:
        row = attention_mask[:, 0, -1, :S]
        valid = row if row.dtype == torch.bool else row == 0
        valid = valid.expand(bsz, S)
        idx = torch.arange(S, device=dev, dtype=torch.int32)
        ends = torch.where(valid, idx + 1, 0).amax(-1)
        starts = torch.minimum(torch.where(valid, idx, S).amin(-1), ends)
        return ends.to(torch.int32).contiguous(), starts.to(torch.int32).contiguous()
    else:
        lens = torch.full((bsz,), S, dtype=torch.int32, device=dev)
    starts = None
    if window is not None:
        starts = torch.clamp(lens - int(window), min=0)
    return lens, starts


def custom_hf_decode_attention_forward(module: torch.nn.Module, query_states: torch.Tensor,
                                       key_states: torch.Tensor, value_states: torch.Tensor,
                                       attention_mask, scaling: float, dropout: float = 0.0, **kwargs):
    """eager_attention_forward replacement: decode steps on the split-KV HIP
    kernels over the dense cache, everything else on transformers' eager path.
    Returns (attn_output [B, Hq, D], None) on decode steps (reshaped by the
    caller exactly as eager's [B, 1, Hq, D])."""
    if query_states.shape[2] == 1:
        source = _range_source(query_states, key_states, attention_mask, kwargs)
        if source is not None:
            return decode_hf(query_states, key_states, value_states, *source, scaling), None
    bounds = _decode_bounds(query_states, key_states, attention_mask, kwargs)
    if bounds is None:
        return native_eager_attention_forward(module, query_states, key_states, value_states,
                                              attention_mask, scaling, dropout, **kwargs)
    lens, starts = bounds
    out = flash_decode_gqa_hf_dense_optimized(query_states.squeeze(2), key_states, value_states, lens, starts,
                                              sm_scale=scaling)
    return out, None


def custom_hf_decode_attention_forward_fp8(module: torch.nn.Module, query_states: torch.Tensor,
                                           key_states: torch.Tensor, value_states: torch.Tensor,
                                           attention_mask, scaling: float, dropout: float = 0.0, **kwargs):
    """FP8 variant: Q, K and V are quantised per call with per-tensor scales
    (the codes of quantize_to_fp8 of their fp32 values, as
    triton_gqa_decode_hf_fp8.py:268-273 takes them); the output keeps the
    query dtype.  16-bit tensors are quantised inside the decode kernels, any
    others (and more than 16 query heads per KV head, where K and V are read
    several times) by a pass of their own."""
    q, k, v = query_states, key_states, value_states
    if (q.shape[2] == 1 and q.dtype in (torch.float16, torch.bfloat16) and k.dtype is q.dtype and v.dtype is q.dtype
            and q.is_cuda and k.is_cuda and v.is_cuda and 0 < q.numel() and 0 < k.numel()
            and q.shape[1] <= 16 * k.shape[1]):
        source = _range_source(q, k, attention_mask, kwargs)
        if source is not None:
            return decode_quantizing_to_fp8(q, k, v, *source, scaling), None
    bounds = _decode_bounds(query_states, key_states, attention_mask, kwargs)
    if bounds is None:
        return native_eager_attention_forward(module, query_states, key_states, value_states,
                                              attention_mask, scaling, dropout, **kwargs)
    lens, starts = bounds
    (q8, sq), (k8, sk), (v8, sv) = quantize_each_to_fp8(query_states.squeeze(2), key_states, value_states)
    out = flash_decode_gqa_hf_fp8(q8, k8, v8, lens, sq, sk, sv, query_states.dtype, start_k_offsets=starts,
                                  sm_scale=scaling)
    return out, None


custom_hf_decode_attention_forward._fsk_patch = True
custom_hf_decode_attention_forward_fp8._fsk_patch = True


def patch_hf_attention(fp8: bool = False, modeling_module=None):
    """Installs the decode attention as ``modeling_module.eager_attention_forward``
    (default: transformers' Qwen3 module) and returns the function it replaced."""
    if modeling_module is None:
        import transformers.models.qwen3.modeling_qwen3 as modeling_module
    prev = modeling_module.eager_attention_forward
    modeling_module.eager_attention_forward = (custom_hf_decode_attention_forward_fp8 if fp8
                                               else custom_hf_decode_attention_forward)
    return prev


@contextlib.contextmanager
def patched_hf_attention(fp8: bool = False, modeling_module=None):
    """Context manager form of patch_hf_attention; restores the previous function."""
    if modeling_module is None:
        import transformers.models.qwen3.modeling_qwen3 as modeling_module
    prev = patch_hf_attention(fp8, modeling_module)
    try:
        yield
    finally:
        modeling_module.eager_attention_forward = prev
