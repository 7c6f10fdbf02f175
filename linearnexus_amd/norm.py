"""Gated RMSNorm output epilogue on MI355X: ``rmsnorm_gated(x, gate, weight, eps)`` computes what the reference's
``FusedRMSNormGated`` module does in its ``__call__`` (linearnexus/modules/linear_attn/kda.py:664-700):
``RMSNorm(x) * weight * sigmoid(gate)`` over the last dimension; ``gate=None`` gives the plain RMSNorm the blocks
use without an output gate (gated_deltanet.py:861-862).  Differentiable with respect to x, gate and weight through
the HIP backward kernel.  There is no other code path: the op raises if the library is missing.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib

Tensor = torch.Tensor


def rmsnorm_gated(x: Tensor, gate: Optional[Tensor], weight: Tensor, eps: float = 1e-5) -> Tensor:
    """``x * rsqrt(mean(x^2, -1) + eps) * weight * sigmoid(gate)`` (kda.py:683-700); ``x, gate [..., d]``, ``weight [d]``."""
    return _lib.host().rmsnorm_gated(x, gate, weight, eps)
