"""Attention over a packed row without the dense bias.

The reference builds ``attn_bias = calculate_attn_bias(...)`` ([B, S, S], 0 / -inf)
and passes it to the model as ``causal_mask`` (src/art/local/train.py:66-73,
177-215, 239-241).  ``packed_attention`` is what a model's attention layer calls
instead of ``softmax(q k^T * scale + attn_bias) v``: same inputs minus the bias,
plus the two id rows the bias was made from.
"""
from __future__ import annotations

from typing import List, Optional

import torch

from . import _lib, ops

ROW_MULTIPLE = 256  # plans cover rows of this granularity; positions past the end see, and are seen by, nothing


def attention_plans(group_ids: torch.Tensor, parent_ids: torch.Tensor) -> List[ops.AttnPlan]:
    """One plan per packed row of ``group_ids`` / ``parent_ids`` ([B, S] int64, the
    PackedTensors rows of src/art/local/pack.py:13-21).  Make them once per
    batch; every layer and head reuses them."""
    if group_ids.dim() == 1:
        group_ids, parent_ids = group_ids.unsqueeze(0), parent_ids.unsqueeze(0)
    return ops.attn_plan_rows(group_ids.contiguous(), parent_ids.contiguous())


def packed_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, plans: List[ops.AttnPlan],
                     scale: Optional[float] = None) -> torch.Tensor:
    """softmax(q k^T * scale + bias) v with the bias of calculate_attn_bias, never built.

    q [B, S, Hq, D], k / v [B, S, Hkv, D] bf16 (any strides over B, S, H; D contiguous;
    a [B, H, S, D] tensor goes in as ``t.transpose(1, 2)``).  Returns [B, S, Hq, D] bf16.
    Differentiable w.r.t. q, k, v."""
    if q.dim() == 3:
        return packed_attention(q.unsqueeze(0), k.unsqueeze(0), v.unsqueeze(0), plans[:1], scale)[0]
    B, S = q.shape[:2]
    if len(plans) < B:
        raise IndexError(f"{len(plans)} plans for {B} rows")
    for plan in plans[:B]:
        if not 0 <= plan.S - S < ROW_MULTIPLE:
            raise ValueError(f"plan made for a row of {plan.S} positions, tensors have {S}")
    first = plans[0]
    if first.rows == B and all(p.batch is first.batch and p.index == b for b, p in enumerate(plans[:B])):
        return _lib.native().attention(q, k, v, first.batch, scale)
    # plans that were made one by one: a call per row
    outs = [_lib.native().attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], plans[b].buf, scale) for b in range(B)]
    return torch.cat(outs, 0)
