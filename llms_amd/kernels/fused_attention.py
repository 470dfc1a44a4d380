"""The attention layer between its two projections on hand-written HIP kernels:
QK-norm, RoPE, the KV-cache write and causal softmax attention.

``attention_core`` runs what ``TritonAttention.forward`` does after the QKV
projection and before ``o`` (reference ``src/kernels/fused_qkv.py:242-282``) as
two or three launches (``llms_amd/csrc/fp_attn.hip``), at the rounding points
of the torch form in ``_eager.py`` and in fp32 between them. It takes bf16
inference on a HIP device with heads of 64 or 128; every other call (other
types and head sizes, gradients, torch.func transforms, autocast, a CPU model)
is the torch form's.

Path: wrapper -> ``torch.ops.llms_amd.attention`` -> C ABI
``fp_attention_bf16`` -> HIP kernels on torch's current stream.
"""

from __future__ import annotations

import torch

from .. import _lib
from ._checks import autocast, plain_norm, transformed


def attention_core(q, k, v, *, q_norm, k_norm, num_heads: int, cache_k, cache_v, cos, sin,
                   start_pos):
    """Attention output ``[B, T, num_heads * D]`` of the flat projections
    ``q [B, T, num_heads * D]``, ``k``, ``v [B, T, kv_heads * D]``, writing the
    new keys and values into ``cache_k``, ``cache_v`` ``[max_batch, kv_heads,
    max_seq, D]`` at ``start_pos`` (an int, or a 0-dim int64 device tensor) ..;
    None, with nothing written, where the kernels do not take the call."""
    if (not q.is_cuda or q.dtype != torch.bfloat16 or cache_k.shape[-1] not in (64, 128)
            or not (plain_norm(q_norm) and plain_norm(k_norm)) or autocast()):
        return None
    if transformed(q, k, v, q_norm.weight, k_norm.weight, cos, sin, cache_k, cache_v):
        return None
    if torch.is_tensor(start_pos):
        pos, start = start_pos, 0
    elif type(start_pos) is int:
        pos, start = None, start_pos
    else:
        return None
    y = _lib.ops().attention(q, k, v, q_norm.weight, k_norm.weight, q_norm.eps, k_norm.eps, cos,
                             sin, cache_k, cache_v, num_heads, start, pos)
    return y if y.dim() == 3 else None
