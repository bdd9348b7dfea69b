"""Transformers attention hook: HIP paged decode when q_len == 1.

Same contract as the reference hook (``runtime/phase2/block_paged_attention.py:24-60``):
registered as ``ALL_ATTENTION_FUNCTIONS["block_paged"]`` with
``config._attn_implementation = "block_paged"`` (``runtime/phase2/worker_server.py:274-281``).
When decode metadata is set, ``q_len == 1`` and the query is on a device, the
fused HIP kernel runs and ``[B, 1, Hq, D]`` is returned (``:37-48``); otherwise
attention on the gathered K/V (prefill, ``:50-60``): one HIP launch for a causal prompt
on the device (``_prefill_kernel_takes``), else the eager chain.

Difference kept on purpose: transformers 5.x hands a custom attention
implementation that has no registered mask function ``attention_mask=None``
(``masking_utils._preprocess_mask_arguments`` returns early for it), so the
reference's eager branch, which only adds a mask when one is given, attends
bidirectionally during prefill. Here a missing mask with ``q_len > 1`` is
replaced by the causal mask (query ``i`` sees keys ``0 .. kv_len - q_len + i``).
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode
from torch.utils._python_dispatch import _get_current_dispatch_mode

from . import _hip
from .paged_attention_hip import _DTYPE_FLAGS, get_paged_decode_batch_metadata, paged_attention_decode_batched


def repeat_kv(hidden_states: torch.Tensor, n_rep: int) -> torch.Tensor:
    if n_rep == 1:
        return hidden_states
    batch, num_key_value_heads, slen, head_dim = hidden_states.shape
    hidden_states = hidden_states[:, :, None, :, :].expand(batch, num_key_value_heads, n_rep, slen, head_dim)
    return hidden_states.reshape(batch, num_key_value_heads * n_rep, slen, head_dim)


def _causal_block(q_len: int, kv_len: int, device: torch.device) -> torch.Tensor:
    """``True`` where query ``i`` (the last ``q_len`` of ``kv_len`` positions) must not see key ``j``."""
    qpos = torch.arange(kv_len - q_len, kv_len, device=device).view(-1, 1)
    return torch.arange(kv_len, device=device).view(1, -1) > qpos


def _rows_aligned(t: torch.Tensor) -> bool:
    """Whether the prefill kernel can read ``t [B, H, T, D]`` with 16-byte loads."""
    b, h, n, _ = t.shape
    sb, sh, sn, unit = t.stride()
    return (unit == 1 and t.data_ptr() % 16 == 0 and (b == 1 or sb % 8 == 0) and (h == 1 or sh % 8 == 0)
            and (n == 1 or sn % 8 == 0))


def _prefill_launch_holds(b: int, hkv: int, groups: int, q_len: int, kv_len: int) -> bool:
    """Whether one launch of ``mx_prefill_attn`` takes these sizes: fewer than 2**32 threads in
    workgroups of 512 (4 units of 32 query rows of a head each), tokens a 32-bit index."""
    workgroups = b * hkv * -(-(-(-q_len // 32) * groups) // 4)
    return workgroups * 512 < 1 << 32 and kv_len <= 1 << 30


def _prefill_kernel_takes(query, key, value, scaling, num_kv_groups) -> bool:
    """Whether ``mx_prefill_attn`` gives this call's causal attention. It takes plain device tensors
    outside autograd, tracing, function transforms and autocast (the eager chain is what those
    see), of one 16-bit dtype and a supported head_dim, with at least as many keys as queries (a
    query before the first key has no visible token: the eager chain's softmax over nothing) and a
    positive scale (the kernel masks scaled scores with -inf) that fp32 holds, also times log2(e)."""
    for t in (query, key, value):
        if type(t) is not torch.Tensor or not t.is_cuda or t.dim() != 4:
            return False
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or torch.is_autocast_enabled("cuda"):
        return False
    if (_get_current_dispatch_mode() is not None or _get_current_function_mode() is not None
            or forward_ad._current_level >= 0):
        return False
    wrapped = torch._C._functorch.is_functorch_wrapped_tensor
    if wrapped(query) or wrapped(key) or wrapped(value):
        return False
    if torch.is_grad_enabled() and (query.requires_grad or key.requires_grad or value.requires_grad):
        return False
    b, hq, q_len, d = query.shape
    _, hkv, kv_len, _ = key.shape
    return (query.dtype in _DTYPE_FLAGS and key.dtype == query.dtype and value.dtype == query.dtype
            and query.device == key.device == value.device
            and value.shape == key.shape and key.shape[0] == b and key.shape[3] == d and d in (64, 128)
            and hkv > 0 and hq == hkv * num_kv_groups and b > 0 and 2 <= q_len <= kv_len
            and isinstance(scaling, (int, float)) and 2.0**-125 <= scaling <= 2.0**126
            and _prefill_launch_holds(b, hkv, num_kv_groups, q_len, kv_len)
            and kv_len * max(key.stride(2), value.stride(2)) < 1 << 31
            and _rows_aligned(query) and _rows_aligned(key) and _rows_aligned(value))


def _prefill(query, key, value, scaling) -> tuple[torch.Tensor, torch.Tensor]:
    """Causal attention of a prompt: ``out [B, P, Hq, D]`` and the weights ``[B, Hq, P, S]``."""
    b, hq, q_len, d = query.shape
    hkv, kv_len = key.shape[1], key.shape[2]
    out = torch.empty((b, q_len, hq, d), dtype=query.dtype, device=query.device)
    weights = torch.empty((b, hq, q_len, kv_len), dtype=query.dtype, device=query.device)

    def strides(t):  # the stride of a dimension of one is never used and may be anything
        (tb, th, tn, _), (sb, sh, sn, _) = t.shape, t.stride()
        return sb if tb > 1 else 0, sh if th > 1 else 0, sn if tn > 1 else 0

    with _hip.on_device(query.device):
        _hip.check(_hip.load().mx_prefill_attn(
            query.data_ptr(), *strides(query), key.data_ptr(), *strides(key), value.data_ptr(), *strides(value), b, hq,
            hkv, q_len, kv_len, d, float(scaling), out.data_ptr(), weights.data_ptr(), _DTYPE_FLAGS[query.dtype],
            _hip.stream_handle(query.device)), "mx_prefill_attn")
    return out, weights


def block_paged_attention_forward(module, query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                                  attention_mask: torch.Tensor | None, scaling: float, dropout: float = 0.0, **kwargs):
    num_kv_groups = getattr(module, "num_key_value_groups", 1)
    meta = get_paged_decode_batch_metadata()
    if meta is not None and query.shape[-2] == 1 and query.is_cuda:
        attn_output = paged_attention_decode_batched(query=query, metadata=meta, num_kv_groups=num_kv_groups,
                                                     scaling=scaling)
        return attn_output.transpose(1, 2).contiguous(), None

    if (attention_mask is None and not (dropout > 0.0 and module.training)
            and _prefill_kernel_takes(query, key, value, scaling, num_kv_groups)):
        return _prefill(query, key, value, scaling)

    key_states = repeat_kv(key, num_kv_groups)
    value_states = repeat_kv(value, num_kv_groups)
    attn_weights = torch.matmul(query, key_states.transpose(2, 3).contiguous()) * scaling
    if attention_mask is not None:
        attn_weights = attn_weights + attention_mask
    elif query.shape[-2] > 1:
        attn_weights = attn_weights.masked_fill(_causal_block(query.shape[-2], key.shape[-2], query.device),
                                                float("-inf"))
    attn_weights = F.softmax(attn_weights, dim=-1, dtype=torch.float32).to(query.dtype)
    if dropout > 0.0 and module.training:
        attn_weights = F.dropout(attn_weights, p=dropout)
    attn_output = torch.matmul(attn_weights, value_states)
    return attn_output.transpose(1, 2).contiguous(), attn_weights


def register_block_paged_attention() -> None:
    """``ALL_ATTENTION_FUNCTIONS.register("block_paged", ...)`` as ``worker_server.py:274-281`` does."""
    from transformers.modeling_utils import ALL_ATTENTION_FUNCTIONS

    ALL_ATTENTION_FUNCTIONS.register("block_paged", block_paged_attention_forward)
