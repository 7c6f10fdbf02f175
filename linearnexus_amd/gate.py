"""Gate activations of the KDA and Gated DeltaNet blocks on MI355X.

``kda_gate(g, A_log, head_k_dim, g_bias=None, beta=None, threshold=20.0)`` mirrors
linearnexus/modules/linear_attn/kda.py:120-172: ``g [B,T,H*dk]`` -> ``-exp(A_log)[h] * softplus(g + g_bias)`` reshaped
to ``[B,T,H,dk]``, plus ``sigmoid(beta)`` in fp32 when ``beta`` is given.  Additive: ``out_dtype`` (default: the
input's dtype, like the reference; ``torch.float32`` feeds ``kda_chunkwise`` without a cast and without rounding the
log-decay to bf16).  Differentiable with respect to g, A_log, g_bias and beta through the HIP kernels; there is no
other code path.

``gated_deltanet_gate(a, A_log, dt_bias, b=None, allow_neg_eigval=False)`` is what the Gated DeltaNet block computes
inline between its projections and the scan (gated_deltanet.py:804-815): ``g = -exp(A_log) * softplus(a + dt_bias)`` and
``beta = sigmoid(b)`` (times 2 with ``allow_neg_eigval``), both ``[..., H]`` in fp32 like the reference's.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib
from .linear_attn import _DT

Tensor = torch.Tensor


def kda_gate(g: Tensor, A_log: Tensor, head_k_dim: int, g_bias: Optional[Tensor] = None, beta: Optional[Tensor] = None,
             threshold: float = 20.0, *, out_dtype: Optional[torch.dtype] = None) -> Tuple[Tensor, Optional[Tensor]]:
    """KDA gate computation (kda.py:120-172): returns ``(g_out [B,T,H,dk], sigmoid(beta) or None)``."""
    if out_dtype is not None and out_dtype not in _DT:
        raise RuntimeError(f"unsupported out_dtype {out_dtype}")
    return _lib.host().kda_gate(g, A_log, head_k_dim, g_bias, beta, threshold, None if out_dtype is None else _DT[out_dtype])


def gated_deltanet_gate(a: Tensor, A_log: Tensor, dt_bias: Optional[Tensor] = None, b: Optional[Tensor] = None,
                        allow_neg_eigval: bool = False) -> Tuple[Tensor, Optional[Tensor]]:
    """Gated DeltaNet's decay gate and learning rate (gated_deltanet.py:804-815): returns ``(g, beta or None)`` in fp32,
    shaped like ``a`` (``[..., H]``: the block's ``[batch, seq, num_v_heads]``, which it then transposes)."""
    return _lib.host().gdn_gate(a, A_log, dt_bias, b, 2.0 if allow_neg_eigval else 1.0)
