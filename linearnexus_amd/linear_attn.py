"""Delta-rule layer ops on MI355X with the reference's signatures.

The nine ops mirror ``linearnexus.modules.linear_attn`` (names, positional order, defaults,
return conventions; linearnexus/modules/linear_attn/__init__.py:15-58): head-first
``[B, H, T, d]`` tensors in, ``(output, final_state)`` out, fp32 state.  Tensors are
``torch`` CUDA tensors (PyTorch only supplies device memory and the stream); every op
launches hand-written gfx950 kernels through the C-ABI and raises if the library is
missing -- there is no other code path.

Differences from the reference, all additive: ``*_step`` take ``inplace=True`` to update
the state buffer in place; the chunk ops take ``cu_seqlens`` for packed variable-length
batches and are differentiable (``torch.autograd``) through the HIP backward kernels.
"""
from __future__ import annotations

import os

from dataclasses import dataclass
from typing import Optional, Tuple

import torch

from . import _lib
from ._lib import LNX_BF16, LNX_F32

Tensor = torch.Tensor
_DT = {torch.float32: LNX_F32, torch.bfloat16: LNX_BF16}
CHUNK = 64  # the kernels' chunk length; results do not depend on it


# --------------------------------------------------------------------------------------
# helpers
# --------------------------------------------------------------------------------------

def _check_inputs(q: Tensor, k: Tensor, v: Tensor) -> None:
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor on an AMD GPU, got {type(t).__name__}")
        if not t.is_cuda:
            raise RuntimeError(f"{name} is on {t.device}; the delta-rule ops run on the GPU only")
    if q.dtype not in _DT:
        raise RuntimeError(f"unsupported dtype {q.dtype}: use float32 or bfloat16")
    if k.dtype != q.dtype or v.dtype != q.dtype:
        raise RuntimeError(f"q, k, v must share one dtype, got {q.dtype}, {k.dtype}, {v.dtype}")
    if q.shape != k.shape or q.shape[:-1] != v.shape[:-1]:
        raise RuntimeError(f"shape mismatch: q {tuple(q.shape)} k {tuple(k.shape)} v {tuple(v.shape)}")


def _f32(t: Tensor) -> Tensor:
    return t.to(torch.float32).contiguous()


def _wants_grad(*tensors) -> bool:
    """The reference's token-by-token ops are differentiable like everything in JAX, and its blocks call them while
    training (sequences of at most 32 tokens, gated_deltanet.py:836-846).  The token kernels have no backward pass;
    when a gradient is wanted the same function is computed by the chunk kernels, which have one."""
    return torch.is_grad_enabled() and any(isinstance(t, torch.Tensor) and t.requires_grad for t in tensors)


def _promote(q: Tensor, k: Tensor, v: Tensor):
    """The reference up-casts q, k, v to float32 whatever they are and returns the output in q's dtype
    (delta_net.py:170-179, :213; gated_deltanet.py:167-175, :229).  The kernels take one dtype, float32 or bfloat16:
    anything else -- mixed dtypes (the DeltaNet block normalises q, k in float32 next to a bf16 v,
    delta_net.py:566-575), float16, float64 -- is computed in float32 and the output cast back to q's dtype.
    Returns (q, k, v, dtype to cast the output to or None)."""
    ts = (q, k, v)
    if not all(isinstance(t, torch.Tensor) and t.is_floating_point() for t in ts):
        return q, k, v, None  # _check_inputs reports it
    if q.dtype == k.dtype == v.dtype and q.dtype in _DT:
        return q, k, v, None
    return q.to(torch.float32), k.to(torch.float32), v.to(torch.float32), q.dtype


def _squeeze_beta(beta: Tensor, ndim: int) -> Tensor:
    # delta_net.py:166-167, :257-258, :378-379 -- a trailing singleton is accepted
    return beta.squeeze(-1) if beta.dim() == ndim else beta


# Test hooks: the tiling overrides of ``lnx_scan_args`` (0 = the library's choice).  The GPU tests set them to reach both
# slab widths of the sequential kernels, and the grouped form of the fp32 output kernel, at small shapes.
_test_hooks = {"scan_slab": 0, "out_slabs": 0}


# --------------------------------------------------------------------------------------
# state caches (delta_net.py:81-118, gated_deltanet.py:72-128, kda.py:57-113)
# --------------------------------------------------------------------------------------

@dataclass
class DeltaNetState:
    """Cache for DeltaNet generation (delta_net.py:81-118): ``S [batch, heads, key_dim, value_dim]`` float32 and the
    conv cache ``[batch, kernel-1, channels]`` of the block's one convolution over the concatenated q, k, v."""
    S: Tensor
    conv_state: Optional[Tensor] = None

    @classmethod
    def zeros(cls, batch_size, num_heads, key_dim, value_dim, conv_channels=None, conv_size=4, *, device="cuda"):
        S = torch.zeros(batch_size, num_heads, key_dim, value_dim, dtype=torch.float32, device=device)
        conv_state = None
        if conv_channels is not None:
            conv_state = torch.zeros(batch_size, conv_size - 1, conv_channels, dtype=torch.float32, device=device)
        return cls(S=S, conv_state=conv_state)


@dataclass
class _GatedState:
    """``S [batch, num_v_heads, key_dim_per_head, value_dim_per_head]`` float32 and one conv cache each for q, k
    (``[batch, kernel-1, key_dim_total]``) and v (``[batch, kernel-1, value_dim]``)."""
    S: Tensor
    conv_state_q: Optional[Tensor] = None
    conv_state_k: Optional[Tensor] = None
    conv_state_v: Optional[Tensor] = None

    @classmethod
    def zeros(cls, batch_size, num_v_heads, key_dim_per_head, value_dim_per_head, key_dim_total=None, value_dim=None,
              conv_size=4, use_conv=True, *, device="cuda"):
        z = lambda *shape: torch.zeros(*shape, dtype=torch.float32, device=device)
        state = cls(S=z(batch_size, num_v_heads, key_dim_per_head, value_dim_per_head))
        if use_conv and key_dim_total is not None and value_dim is not None:
            state.conv_state_q = z(batch_size, conv_size - 1, key_dim_total)
            state.conv_state_k = z(batch_size, conv_size - 1, key_dim_total)
            state.conv_state_v = z(batch_size, conv_size - 1, value_dim)
        return state


@dataclass
class GatedDeltaNetState(_GatedState):
    """Cache for Gated DeltaNet generation (gated_deltanet.py:72-128)."""


@dataclass
class KDAState(_GatedState):
    """Cache for KDA generation (kda.py:57-113)."""


# --------------------------------------------------------------------------------------
# single-token decode step
# --------------------------------------------------------------------------------------

def _step(q, k, v, g, beta, state, scale, l2norm, o_dtype_from_state, inplace):
    # contiguous inputs of one kernel dtype with fp32 beta, g and state and no gradient wanted: a decode loop's calls
    out = _lib.host().step(q, k, v, g, beta, state, scale, l2norm, o_dtype_from_state, inplace)
    return _step_general(q, k, v, g, beta, state, scale, l2norm, o_dtype_from_state, inplace) if out is None else out


def _step_general(q, k, v, g, beta, state, scale, l2norm, o_dtype_from_state, inplace):
    q, k, v, back = _promote(q, k, v)
    if back is not None:
        o, s_out = _step(q, k, v, g, beta, state, scale, l2norm, o_dtype_from_state, inplace)
        return (o if o_dtype_from_state else o.to(back)), s_out
    _check_inputs(q, k, v)
    if q.dim() != 3:
        raise RuntimeError(f"step ops take [B, H, d] vectors, got q {tuple(q.shape)}")
    beta = _squeeze_beta(beta, 3)
    if _wants_grad(q, k, v, g, beta, state):
        if inplace:
            raise RuntimeError("inplace=True overwrites the state a backward pass would need")
        # the token kernels normalise and compute in fp32 (gated_deltanet.py:193-195): so does this path, so that the
        # values do not depend on whether a gradient is wanted
        up = (lambda t: t.to(torch.float32)) if (l2norm and q.dtype != torch.float32) else (lambda t: t)
        o, s_out = _chunk(up(q)[:, :, None], up(k)[:, :, None], up(v)[:, :, None], None if g is None else g[:, :, None],
                          beta[:, :, None], scale, state, CHUNK, l2norm,
                          torch.float32 if (o_dtype_from_state or l2norm) else q.dtype, False, None)
        return o[:, :, 0].to(state.dtype if o_dtype_from_state else q.dtype), s_out
    B, H, dk = q.shape
    dv = v.shape[-1]
    if g is not None and tuple(g.shape) not in ((B, H), (B, H, dk)):
        raise RuntimeError(f"gate shape {tuple(g.shape)} matches neither {(B, H)} nor {(B, H, dk)}")
    if tuple(beta.shape) != (B, H):
        raise RuntimeError(f"beta shape {tuple(beta.shape)} != {(B, H)}")
    if tuple(state.shape) != (B, H, dk, dv):
        raise RuntimeError(f"state shape {tuple(state.shape)} != {(B, H, dk, dv)}")
    if inplace and (state.dtype != torch.float32 or not state.is_contiguous()):
        raise RuntimeError("inplace=True needs a contiguous float32 state")
    out = _lib.host().step(q.contiguous(), k.contiguous(), v.contiguous(), None if g is None else _f32(g), _f32(beta),
                           _f32(state), scale, l2norm, o_dtype_from_state, inplace)
    if out is None:
        raise RuntimeError("beta, g and state must be on the GPU of q, k and v")
    return out


def delta_rule_step(q, k, v, beta, state, scale=None, *, inplace=False) -> Tuple[Tensor, Tensor]:
    """One decode token of plain DeltaNet (delta_net.py:357-397)."""
    return _step(q, k, v, None, beta, state, scale, False, False, inplace)


def gated_delta_rule_step(q, k, v, g, beta, state, scale=None, use_qk_l2norm=True, *, inplace=False):
    """One decode token of Gated DeltaNet, ``g [B,H]`` (gated_deltanet.py:539-597)."""
    return _step(q, k, v, g, beta, state, scale, use_qk_l2norm, False, inplace)


def kda_step(q, k, v, g, beta, state, scale=None, use_qk_l2norm=True, *, inplace=False):
    """One decode token of KDA, ``g [B,H,dk]``; output in the state's dtype (kda.py:286-347)."""
    return _step(q, k, v, g, beta, state, scale, use_qk_l2norm, True, inplace)


# --------------------------------------------------------------------------------------
# token-by-token scan
# --------------------------------------------------------------------------------------

def _check_cu_seqlens(cu, T: int) -> Tensor:
    """``cu_seqlens`` as an integer tensor.  A table that lives on the host (list, numpy array, CPU tensor) is
    validated here: one-dimensional, at least two entries, ``cu[0] == 0``, non-decreasing, ``cu[-1] == T`` -- every
    token belongs to exactly one sequence; anything else raises ``ValueError``.  A table that is already on the GPU is
    not read back (that would synchronise the stream): the kernels clamp its entries to ``[0, T]`` and treat a
    decreasing pair as an empty sequence, so a malformed table cannot send them outside the tensors, but tokens it
    does not cover then keep unspecified outputs and gradients."""
    if not isinstance(cu, torch.Tensor):
        cu = torch.as_tensor(cu)
    if cu.is_floating_point() or cu.dim() != 1 or cu.numel() < 2:
        raise ValueError(f"cu_seqlens must be a 1-D integer table with at least two entries, got shape {tuple(cu.shape)} {cu.dtype}")
    if not cu.is_cuda:
        c = cu.to(torch.int64)
        if int(c[0]) != 0 or int(c[-1]) != T or bool((c[1:] < c[:-1]).any()):
            raise ValueError(f"cu_seqlens must start at 0, never decrease and end at T = {T}; got {c.tolist()[:8]}"
                             f"{' ...' if c.numel() > 8 else ''} (last {int(c[-1])})")
    return cu


def _packed_table(cu_seqlens, q: Tensor) -> Optional[Tensor]:
    """The checked table as the kernels read it: int32 on q's device."""
    if cu_seqlens is None:
        return None
    return _check_cu_seqlens(cu_seqlens, q.shape[2]).to(device=q.device, dtype=torch.int32).contiguous()


def _recurrent(q, k, v, g, beta, scale, initial_state, l2norm, cu_seqlens=None):
    q, k, v, back = _promote(q, k, v)
    if back is not None:
        o, sT = _recurrent(q, k, v, g, beta, scale, initial_state, l2norm, cu_seqlens)
        return o.to(back), sT
    if _wants_grad(q, k, v, g, beta, initial_state):
        if l2norm and q.dtype != torch.float32:  # fp32 normalisation and arithmetic, like the token kernels
            o, sT = _chunk(q.to(torch.float32), k.to(torch.float32), v.to(torch.float32), g, beta, scale, initial_state, CHUNK,
                           l2norm, torch.float32, False, cu_seqlens)
            return o.to(q.dtype), sT
        return _chunk(q, k, v, g, beta, scale, initial_state, CHUNK, l2norm, q.dtype, False, cu_seqlens)
    cu = None if cu_seqlens is None else _packed_table(cu_seqlens, q)
    return _lib.host().recurrent(q, k, v, g, beta, initial_state, scale, l2norm, cu)


def delta_rule_recurrent(q, k, v, beta, initial_state=None, scale=None, backend=None, *, cu_seqlens=None):
    """Token-by-token DeltaNet scan in fp32 (delta_net.py:126-213)."""
    return _recurrent(q, k, v, None, beta, scale, initial_state, False, cu_seqlens)


def gated_delta_rule_recurrent(q, k, v, g, beta, scale=None, initial_state=None, use_qk_l2norm=True, *,
                               cu_seqlens=None):
    """Token-by-token Gated DeltaNet scan, ``g [B,H,T]`` (gated_deltanet.py:136-229)."""
    return _recurrent(q, k, v, g, beta, scale, initial_state, use_qk_l2norm, cu_seqlens)


def kda_recurrent(q, k, v, g, beta, scale=None, initial_state=None, use_qk_l2norm=True, *, cu_seqlens=None):
    """Token-by-token KDA scan, ``g [B,H,T,dk]`` (kda.py:179-283)."""
    return _recurrent(q, k, v, g, beta, scale, initial_state, use_qk_l2norm, cu_seqlens)


# --------------------------------------------------------------------------------------
# chunked scan (forward + backward)
# --------------------------------------------------------------------------------------

def l2norm_rows(x: Tensor) -> Tensor:
    """``x / (|x|_2 + 1e-6)`` over the last dimension, in x's dtype (gated_deltanet.py:273-275; what the DeltaNet
    block applies to q and k before the op, delta_net.py:566-575).  Differentiable."""
    return _lib.host().l2norm(x)


def _l2norm_rows_bwd(x: Tensor, dy: Tensor) -> Tensor:
    return _lib.host().l2norm_bwd(x, dy)


def _chunk_forward(q, k, v, g, beta, initial_state, scale, l2norm, o_dtype, cu_seqlens, forward_only,
                   raw_gate=None):
    """One chunked scan, ``(o, final_state)``.  Without ``forward_only`` the call is a node of the autograd graph
    whose backward is lnx_chunk_bwd; with it the kernels skip what only a backward pass reads.  ``raw_gate = (A_log, g_bias or None,
    threshold)``: ``g`` is the raw per-channel gate projection in q's dtype and the kernels apply kda_gate's
    activation themselves."""
    A_log, g_bias, threshold = raw_gate or (None, None, 0.0)
    return _lib.host().chunk(q, k, v, g, beta, initial_state, scale, l2norm, _DT[o_dtype], _packed_table(cu_seqlens, q),
                             forward_only, A_log, g_bias, threshold,
                             _test_hooks["scan_slab"], _test_hooks["out_slabs"])


_CHUNK_DK = (64, 128, 256)  # key head dimensions the chunk kernels are built for


def _prefill_segments(B: int, H: int, T: int, dv: int, dk: int = 256, two_byte: bool = True, vector_gate: bool = False) -> int:
    """How many segments a forward-only call is cut into (1: not at all).  The sequential kernels have one workgroup
    per (batch, head, 32 or 64 value columns); a few long prompts leave most of the 256 CUs without one.  Segments are run
    as independent sequences -- see _segmented_forward -- which is three times the scan work over nseg times the
    workgroups and one short step per segment.  LNX_PREFILL_SEGMENTS forces a count (0 or 1: never).

    dk <= 128: the first pass has w = B H (dk + dv) / 64 workgroups per segment, so 256 / w segments fill the chip once.
    Segments of 16 chunks or more, but eight of them where the chip has room (a segment's step costs as much as two chunks).
    bf16 d128 unless said, one chain -> cut, on the kernels as they are: 4 heads of 4096 tokens 85 -> 59 us, of 16384 306 -> 103; 16 heads
    (w = 64) of 8192 174 -> 124, of 32768 690 -> 385 in eight segments (four: 422).  The kernels that form W and U prepare both passes: fp32 4
    heads of 4096 275 -> 175, bf16 per-channel gate 4 heads of 8192 185 -> 130 (4096: 103 -> 111, so not), w = 64 never (8192: 289 -> 346).
    The lines were drawn on a slower first pass: what lies before them would often gain, too, at w <= 32 from 48 chunks on (4 heads of 3072 tokens 67 -> 54; 2048: 49 -> 49), at w = 64 from 64 on (4096 tokens 93 -> 80; 3072: 73 ->
    71), past w = 64 from 128 on at d64 (40 heads of 8192 tokens 164 -> 140) and from 256 on at d128 (20 heads of 16384 351 -> 311).

    dk = 256, and rows that would have to be copied to become heads: at most an eighth of the CUs busy and every segment keeps >= 64 chunks
    (fewer heads of 512 values gain less than their longer preparation costs: 16 workgroups of 4096 tokens 196 -> 216 us)."""
    forced = os.environ.get("LNX_PREFILL_SEGMENTS")
    chunks = -(-T // CHUNK)
    if forced is not None:
        return max(1, min(int(forced), chunks))
    if dk > 128:
        wide = B * H * -(-dv // 64)
        if wide > 32 or T < 16384 * max(1, wide // 16):  # measured: no gain at 32 workgroups x 16384 tokens, loss at 64
            return 1
        return max(1, min(256 // wide, T // 4096))
    direct = two_byte and not vector_gate
    w = B * H * (-(-dk // 64) + -(-dv // 64))
    if w > (64 if direct else 32) or chunks < (64 if (direct and w <= 32) or not two_byte else 128):
        return 1
    return min((512 if w > 32 and chunks >= 512 else 256) // w, max(8, chunks // 16))


def _prefill_segments_256(B: int, H: int, T: int, dv: int) -> int:
    """The same for dk = 256 in bf16 without a per-channel gate, where the first pass forms no outputs and the second finds everything prepared.
    A chain takes 2.5 us a chunk (3.3 when the lines were drawn), cutting costs a setup and a short step per segment.  One chain -> cut, us:
    w <= 64 (H4 dv 512, w = 48) 3072 tokens 133 -> 119, 4096 171 -> 149, 8192 333 -> 196; w <= 128 (H8 dv 512, w = 96) 4096 175 -> 165, 8192 338 ->
    258 (2048: 94 -> 119, so not); never beyond (H12 dv 512, w = 144: 8192 tokens 352 -> 450 and more).  Between 32 and some 40 chunks the cut now
    loses (2048 tokens, w = 12 94 -> 98, w = 48 95 -> 102, w = 64 94 -> 104).  Eight segments; four where w or a short prompt leaves them too little
    (w = 96, 8192 tokens: 258 against 300; they would be the better choice up to 96 chunks at w = 48, too: 4096 tokens 137 against 149), sixteen of
    few heads and long prompts (w = 5, 32768 tokens: 284 against 348; w = 48: 544 against 484)."""
    chunks, w = -(-T // CHUNK), B * H * (4 + -(-dv // 64))
    if os.environ.get("LNX_PREFILL_SEGMENTS") is not None:
        return _prefill_segments(B, H, T, dv)
    if w > 128 or chunks < (32 if w <= 64 else 64):
        return 1
    return 4 if w > 64 or chunks < 64 else 16 if w <= 24 and chunks >= 256 else 8


def _segmented_forward(q, k, v, g, beta, scale, initial_state, l2norm, o_dtype, nseg):
    """Forward pass of a long sequence as nseg segments processed in parallel (no gradients).

    The scan is linear in the state: over a segment s, S_out = A_s S_in + B_s with A_s [dk, dk] the product of the
    segment's token transitions and B_s [dk, dv] what the segment writes into a zero state.  One pass with the
    value columns extended to [v | 0] and every segment started from [0 | I] leaves [B_s | A_s] as its final states;
    a short kernel chains the segments' entering states; a second pass with those as initial states gives the
    outputs.  (The same (A_s, B_s) pair is what ranks would exchange if a sequence were split across GPUs.)"""
    return _lib.host().chunk_segmented(q, k, v, g, _squeeze_beta(beta, 4), initial_state, scale, l2norm, _DT[o_dtype], nseg)


def _chunk(q, k, v, g, beta, scale, initial_state, chunk_size, l2norm, o_dtype, need_mult16, cu_seqlens):
    if need_mult16 and chunk_size % 16 != 0:
        # gated_deltanet.py:318-320, kda.py:438-440
        raise ValueError(f"chunk_size (BT={chunk_size}) must be divisible by BC=16.")
    if chunk_size <= 0:
        raise ValueError(f"chunk_size must be positive, got {chunk_size}")
    if scale is None:
        scale = q.shape[-1] ** -0.5
    q, k, v, back = _promote(q, k, v)
    if back is not None:  # computed in float32; o_dtype is what the caller gets
        o, sT = _chunk(q, k, v, g, beta, scale, initial_state, chunk_size, l2norm, torch.float32, need_mult16, cu_seqlens)
        return o.to(o_dtype), sT
    dk, dv = q.shape[-1], v.shape[-1]
    dkp = next((c for c in _CHUNK_DK if dk <= c), None)
    dvp = -(-dv // 64) * 64
    forward_only = not _wants_grad(q, k, v, g, beta, initial_state)
    if dkp is None or q.dim() != 4 or (dkp, dvp) == (dk, dv):
        if forward_only and dkp is not None and q.dim() == 4 and cu_seqlens is None:
            # batch rows become heads: free for contiguous tensors, a copy of the token-first views of several rows
            folds = q.shape[0] == 1 or (q.is_contiguous() and k.is_contiguous() and v.is_contiguous())
            two_byte, vector_gate = q.element_size() == 2, g is not None and g.dim() == 4 and g.shape[-1] == dk
            if folds and dk > 128 and two_byte and not vector_gate:
                nseg = _prefill_segments_256(q.shape[0], q.shape[1], q.shape[2], dv)
            else:
                nseg = _prefill_segments(q.shape[0], q.shape[1], q.shape[2], dv, dk if folds else 256, two_byte, vector_gate)
            if nseg > 1:
                return _segmented_forward(q, k, v, g, beta, scale, initial_state, l2norm, o_dtype, nseg)
        return _chunk_forward(q, k, v, g, beta, initial_state, scale, l2norm, o_dtype, cu_seqlens, forward_only=forward_only)[:2]
    # Head dimensions between the kernels' sizes (the reference's own tests use dk = 8, 16, dv = 8, 32):
    # zero channels are exact.  A zero key/query channel adds nothing to any <q,k>, <k,k> or |x|_2, the state rows
    # and columns it would feed stay zero, and the padded value columns are independent of the others; autograd
    # slices the gradients back.  `scale` was fixed above from the true dk.
    pad = torch.nn.functional.pad
    q, k, v = pad(q, (0, dkp - dk)), pad(k, (0, dkp - dk)), pad(v, (0, dvp - dv))
    if g is not None and g.dim() == 4 and g.shape[-1] == dk:
        g = pad(g, (0, dkp - dk))
    if initial_state is not None:
        initial_state = pad(initial_state, (0, dvp - dv, 0, dkp - dk))
    o, sT = _chunk_forward(q, k, v, g, beta, initial_state, scale, l2norm, o_dtype, cu_seqlens, forward_only=forward_only)[:2]
    return o[..., :dv], sT[..., :dk, :dv]


def delta_rule_chunkwise(q, k, v, beta, initial_state=None, chunk_size=64, scale=None, backend=None, *,
                         cu_seqlens=None):
    """Chunked (WY) DeltaNet scan (delta_net.py:216-354).  ``chunk_size`` is validated and then
    ignored: the kernels always use 64-token chunks, which the result does not depend on."""
    return _chunk(q, k, v, None, beta, scale, initial_state, chunk_size, False, q.dtype, False, cu_seqlens)


def gated_delta_rule_chunkwise(q, k, v, g, beta, scale=None, initial_state=None, chunk_size=64,
                               use_qk_l2norm=True, *, cu_seqlens=None):
    """Chunked Gated DeltaNet scan, ``g [B,H,T]`` (gated_deltanet.py:232-534)."""
    return _chunk(q, k, v, g, beta, scale, initial_state, chunk_size, use_qk_l2norm, q.dtype, True, cu_seqlens)


def kda_chunkwise(q, k, v, g, beta, scale=None, initial_state=None, chunk_size=64, use_qk_l2norm=True, *,
                  cu_seqlens=None, output_dtype=torch.float32):
    """Chunked KDA scan, ``g [B,H,T,dk]`` (kda.py:350-655).  Like the reference, the output is
    float32 whatever the input dtype (kda.py:416, :655); pass ``output_dtype`` to change that."""
    return _chunk(q, k, v, g, beta, scale, initial_state, chunk_size, use_qk_l2norm, output_dtype, True, cu_seqlens)


def kda_chunkwise_raw_gate(q, k, v, g_raw, beta, A_log, g_bias=None, scale=None, initial_state=None, chunk_size=64,
                           use_qk_l2norm=True, *, threshold=20.0, cu_seqlens=None, output_dtype=torch.float32):
    """``kda_gate`` (kda.py:120-172) and ``kda_chunkwise`` (kda.py:350-655) as one op: the KDA block's two steps between
    its projections and its output norm without the fp32 log-decay tensor in between.

    ``g_raw [B,H,T,dk]`` is the raw gate projection in q's dtype -- the block's ``[B,T,H*dk]`` viewed as
    ``[B,T,H,dk].transpose(1, 2)`` is used in place, like q, k, v; ``A_log [H]``, ``g_bias [H*dk]`` as in ``kda_gate``.
    Equal to ``kda_chunkwise(q, k, v, kda_gate(g_raw, A_log, dk, g_bias, out_dtype=float32)[0], beta, ...)`` with the
    activation computed in fp32 inside the chunk kernels; differentiable with respect to q, k, v, g_raw, beta,
    initial_state, A_log and g_bias.  dk must be 64, 128 or 256 and dv a multiple of 64."""
    if chunk_size % 16 != 0:
        raise ValueError(f"chunk_size (BT={chunk_size}) must be divisible by BC=16.")  # kda.py:438-440
    if q.dim() != 4 or q.shape[-1] not in _CHUNK_DK or v.shape[-1] % 64 != 0:
        raise RuntimeError(f"kda_chunkwise_raw_gate needs [B,H,T,d] inputs with dk in {_CHUNK_DK} and dv % 64 == 0, "
                           f"got q {tuple(q.shape)}, v {tuple(v.shape)}")
    if not (q.dtype == k.dtype == v.dtype == g_raw.dtype) or q.dtype not in _DT:
        raise RuntimeError("q, k, v and g_raw must share one of the dtypes float32 / bfloat16")
    if tuple(g_raw.shape) != tuple(q.shape):
        raise RuntimeError(f"g_raw {tuple(g_raw.shape)} must have q's shape {tuple(q.shape)}")
    H, dk = q.shape[1], q.shape[-1]
    if tuple(A_log.shape) != (H,) or (g_bias is not None and tuple(g_bias.shape) != (H * dk,)):
        raise RuntimeError(f"A_log must be [{H}] and g_bias [{H * dk}]")
    if scale is None:
        scale = dk ** -0.5
    return _chunk_forward(q, k, v, g_raw, beta, initial_state, scale, use_qk_l2norm, output_dtype, cu_seqlens,
                          forward_only=not _wants_grad(q, k, v, g_raw, beta, initial_state, A_log, g_bias),
                          raw_gate=(A_log, g_bias, float(threshold)))[:2]
