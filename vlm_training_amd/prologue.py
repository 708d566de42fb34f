"""The element-wise work either side of the attention operator, fused into single passes over HBM.

``qk_norm_rope``  replaces, in the reference's attention layers, ``q_norm(q)``/``k_norm(k)`` (F.rms_norm per
head), the transpose to (B, H, S, D), ``apply_rope``, the transpose back and the ``.contiguous()`` copies
(models/qwen3_vl/model.py:256-269; models/qwen3_5/model.py:110-129 with OffsetRMSNorm and a partial
rotary width): the projections' outputs go in as (T, H, D) *views* (any token / head stride, so the q
half of Qwen3.5's interleaved ``[q | gate]`` projection is read in place), the packed (T, H, D) tensors
the attention operator wants come out.  ``sigmoid_gate`` is ``out * torch.sigmoid(gate)``
(models/qwen3_5/model.py:135).  Both are autograd nodes in csrc/dsa_host.cpp over the C ABI;
there is no fallback path.
"""
from __future__ import annotations

import torch

from . import _lib


@torch.compiler.disable
def qk_norm_rope(q, k, q_weight, k_weight, cos, sin, eps: float = 1e-6, offset: bool = False):
    """q (T, Hq, D), k (T, Hkv, D) bf16 views -> rope(rms_norm(q)), rope(rms_norm(k)) as contiguous (T, H, D).

    ``offset=True`` scales by ``1 + weight`` (OffsetRMSNorm).  cos, sin: (T, R) or (1, T, R), R <= D a
    multiple of 16 (elements past R pass through unrotated)."""
    return tuple(_lib.host().qk_norm_rope(q, k, q_weight, k_weight, cos, sin, float(eps), bool(offset)))


@torch.compiler.disable
def sigmoid_gate(x, gate):
    """``x * torch.sigmoid(gate)`` for x (T, H, D) contiguous and gate a (T, H, D) view (strided allowed)."""
    return _lib.host().sigmoid_gate(x, gate)
