"""RWKV-7's diagonal-plus-low-rank delta rule on MI355X behind the reference's op names.

``dplr_delta_rule_recurrent(q, k, v, a, b, gk, scale=1.0, initial_state=None)`` and
``dplr_delta_rule_step(q, k, v, a, b, gk, state, scale=1.0)`` mirror
linearnexus/modules/linear_attn/rwkv7.py:114-265 (names, positional order, defaults, ``(output, state)`` returns,
output in ``q.dtype``, fp32 state).  Heads of 64 x 64 -- RWKV-7's own -- with at least 16 tokens run over chunks of 64
tokens on the fp32 matrix cores (csrc/dplr_chunk.hip; the reference has no chunked form of this recurrence), anything else
token by token (csrc/dplr.hip).  Both take any gate: a large negative one, down to -inf, ends a document inside a row.
Both ops are differentiable with respect to q, k, v, a, b, gk and the state, as the reference's are under jax.grad (its
RWKV-7 block trains through the scan).  Between the two passes the chunked scan keeps 48 KB per chunk of a (batch, head)
row, as much again as a bf16 call's inputs; the token kernels keep nothing and recompute the states from checkpoints.
Additive: ``dplr_delta_rule_step(..., inplace=True)`` updates the state buffer in place (not differentiable).  There
is no other code path: the ops raise if the library is missing.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib

Tensor = torch.Tensor


def dplr_delta_rule_recurrent(q: Tensor, k: Tensor, v: Tensor, a: Tensor, b: Tensor, gk: Tensor, scale: float = 1.0,
                              initial_state: Optional[Tensor] = None) -> Tuple[Tensor, Tensor]:
    """DPLR scan over ``[B,H,T,.]`` tensors (rwkv7.py:114-213)."""
    return _lib.host().dplr(q, k, v, a, b, gk, scale, initial_state)


def dplr_delta_rule_step(q: Tensor, k: Tensor, v: Tensor, a: Tensor, b: Tensor, gk: Tensor, state: Tensor,
                         scale: float = 1.0, *, inplace: bool = False) -> Tuple[Tensor, Tensor]:
    """One decode token of the DPLR rule on ``[B,H,.]`` vectors (rwkv7.py:216-265)."""
    return _lib.host().dplr_step(q, k, v, a, b, gk, state, scale, inplace)
