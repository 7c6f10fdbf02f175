"""Gradients of bf16 chunk calls whose tokens have next to no beta: between the reverse scan and the chunk-local kernel a row is dv = beta dR,
which says nothing of a token with beta = 0 (padding), so rows below 2^-24 take another way (LNX_BETA_MIN, csrc/chunk_common.h)."""
import numpy as np
import pytest
import torch

from conftest import max_rel
from oracle.adjoint import delta_rule_adjoint
from oracle.inputs import make_inputs, to_bf16_grid

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grads(x, gate, cu=None, token_first=False):
    import linearnexus_amd as la
    lay = (lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)) if token_first else (lambda t: t)
    leaves = {n: lay(torch.from_numpy(x[n]).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32)).requires_grad_(True)
              for n in ("q", "k", "v", "beta", "g", "S0") if n in x}
    q, k, v, beta, s0 = (leaves[n] for n in ("q", "k", "v", "beta", "S0"))
    cu_t = None if cu is None else torch.from_numpy(cu).to(DEV)
    if gate == "none":
        o, S = la.delta_rule_chunkwise(q, k, v, beta, s0, cu_seqlens=cu_t)
    else:
        op = la.gated_delta_rule_chunkwise if gate == "scalar" else la.kda_chunkwise
        o, S = op(q, k, v, leaves["g"], beta, None, s0, 64, False, cu_seqlens=cu_t)
    grads = torch.autograd.grad([o, S], list(leaves.values()), [torch.from_numpy(x["dO"]).to(DEV).to(o.dtype), torch.from_numpy(x["dS"]).to(DEV)])
    return {"d" + ("S0" if n == "S0" else n): t.float().cpu().numpy() for n, t in zip(leaves, grads)}


def _inputs(gate, shape, which):
    x = make_inputs(91, *shape, gate=gate, with_state=True, with_grad=True)
    for n in ("q", "k", "v", "dO"):
        x[n] = to_bf16_grid(x[n])
    rng = np.random.default_rng(3)
    b = x["beta"]
    if which == "some":
        b[rng.random(b.shape) < 0.3] = 0.0
    elif which == "all":
        b[:] = 0.0
    else:  # both sides of the limit, and either sign
        b[:] = np.where(rng.random(b.shape) < 0.7, np.exp2(rng.uniform(-30, 0, b.shape)) * rng.choice([-1, 1], b.shape), b)
        b[..., :3] = [2.0**-24, -(2.0**-24), 2.0**-24 * (1 - 2.0**-20)]
    return x


@pytest.mark.parametrize("which", ["some", "all", "limit"])
@pytest.mark.parametrize("gate,dk,dv", [("none", 64, 64), ("none", 128, 128), ("scalar", 64, 128), ("scalar", 128, 96), ("scalar", 256, 64), ("none", 256, 160),
                                        ("vector", 64, 64), ("vector", 128, 128)])
def test_gradients_with_small_beta(gate, dk, dv, which):
    x = _inputs(gate, (1, 2, 150, dk, dv), which)
    ref = delta_rule_adjoint(x["q"], x["k"], x["v"], x["beta"], x["dO"], x.get("g"), x["dS"], None, x["S0"], False)
    got = _grads(x, gate, token_first=which == "limit")
    errs = {n: max_rel(got[n], ref[n]) if np.abs(ref[n]).max() > 0 else float(np.abs(got[n]).max()) for n in got}
    assert all(e < 2e-2 for e in errs.values()), errs
    # a token's dv carries its beta: relative to its own row, so that no factor went missing; exactly zero without beta
    dv_, r = got["dv"], ref["dv"]
    assert (dv_[x["beta"] == 0] == 0).all()
    rows = np.abs(r).max(-1)
    assert (np.abs(dv_ - r).max(-1)[rows > 1e-30] < 0.1 * rows[rows > 1e-30]).all()


@pytest.mark.parametrize("gate", ["none", "scalar", "vector"])
def test_packed_gradients_with_small_beta(gate):
    x = _inputs(gate, (1, 2, 300, 128, 128), "some")
    cu = np.array([0, 70, 70, 201, 300], np.int32)
    x["S0"] = np.repeat(x["S0"], 4, 0) * np.arange(1, 5, dtype=np.float32)[:, None, None, None]
    x["dS"] = np.repeat(x["dS"], 4, 0)
    got = _grads(x, gate, cu)
    for i, (a, b) in enumerate(zip(cu[:-1], cu[1:])):
        if a == b:
            continue
        s = {n: np.ascontiguousarray(x[n][:, :, a:b]) for n in ("q", "k", "v", "beta", "dO", "g") if n in x}
        ref = delta_rule_adjoint(s["q"], s["k"], s["v"], s["beta"], s["dO"], s.get("g"), x["dS"][i:i + 1], None, x["S0"][i:i + 1], False)
        for n in ("dq", "dk", "dv", "dbeta") + (("dg",) if gate != "none" else ()):
            assert max_rel(got[n][:, :, a:b], ref[n]) < 2e-2, (n, i)
