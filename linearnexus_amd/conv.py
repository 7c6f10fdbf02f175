"""Short causal depthwise convolution (+ fused SiLU) on MI355X behind the reference's helper name.

``depthwise_conv1d_causal(inputs, weight, bias, *, cache=None)`` mirrors linearnexus/core/conv.py:13-68:
``inputs [B,T,D]``, ``weight [K,D]`` (K <= 4), ``bias [D]`` or None, ``cache [B,K-1,D]`` or None; returns
``(output, new_cache)``.  Additive: ``activation="silu"`` fuses the SiLU the blocks apply right after
(gated_deltanet.py:765-779), ``inplace_cache=True`` writes the new cache over the old one (decode) and
``cu_seqlens`` makes the batch packed (``inputs [1,T,D]``: the taps stop at the start of each sequence, as if
every sequence went through the function on its own with a zero cache -- the layout the chunk ops take).
Differentiable with respect to inputs, weight, bias and the carry-in cache through the HIP backward kernels.
There is no other code path: the ops raise if the library is missing.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib
from .linear_attn import _check_cu_seqlens

Tensor = torch.Tensor
_ACT = {None: 0, "none": 0, "silu": 1}


def depthwise_conv1d_causal(inputs: Tensor, weight: Tensor, bias: Optional[Tensor] = None, *,
                            cache: Optional[Tensor] = None, activation: Optional[str] = None,
                            inplace_cache: bool = False, cu_seqlens=None) -> Tuple[Tensor, Tensor]:
    """Depthwise causal conv1d with optional cache warm-start (linearnexus/core/conv.py:13-68)."""
    if activation not in _ACT:
        raise ValueError(f"activation must be None or 'silu', got {activation!r}")
    cu = None
    if cu_seqlens is not None:
        cu = _check_cu_seqlens(cu_seqlens, inputs.shape[1]).to(device=inputs.device, dtype=torch.int32).contiguous()
    return _lib.host().conv1d(inputs, weight, bias, cache, _ACT[activation], inplace_cache, cu)
