"""The chunked RWKV-7 scan (heads of 64 x 64) against the fp64 oracle and its adjoint: lengths around one chunk, decays of
RWKV-7's range, decays so strong that a block's pairs are evaluated one by one, both in one sequence, and growth; 1e-4
(fp32) / 2e-2 (bf16) of max|ref|.  Windows: a call whose work areas are cut into windows of chunks returns the bits of a
call on some of its rows alone."""
import numpy as np
import pytest
import torch

from oracle import dplr as od
from oracle.inputs import to_bf16_grid
from conftest import max_rel

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAMES = ("q", "k", "v", "a", "b", "gk")


def _data(seed, B, H, T, decay, bf16):
    r = np.random.default_rng(seed)
    n = lambda *s: r.standard_normal(s).astype(np.float32)
    d = 64
    kk = n(B, H, T, d)
    kk /= np.linalg.norm(kk, axis=-1, keepdims=True)
    rate = r.random((B, H, T, d)).astype(np.float32)
    gk = {"rwkv": -0.6065 * rate, "none": 0 * rate, "strong": -6 * rate, "growth": 0.01 * rate}.get(decay)
    if decay == "mixed":  # such blocks only where a few channels decay strongly, from the second chunk on
        gk = -0.3 * rate
        gk[:, :, 64:, ::17] -= 9.0
    x = dict(q=n(B, H, T, d), k=n(B, H, T, d) * 0.5, v=n(B, H, T, d), a=-kk, b=kk * r.random((B, H, T, d)).astype(np.float32), gk=gk.astype(np.float32),
             h0=n(B, H, d, d) * 0.5, dO=n(B, H, T, d), dS=n(B, H, d, d) * 0.3)
    if bf16:
        for m in ("q", "k", "v", "a", "b", "dO"):
            x[m] = to_bf16_grid(x[m])
    return x


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("decay,T", [("rwkv", 16), ("rwkv", 63), ("rwkv", 64), ("rwkv", 65), ("rwkv", 330), ("none", 130), ("strong", 100), ("mixed", 200), ("growth", 129)])
def test_scan_and_gradients_match_oracle(decay, T, bf16):
    import linearnexus_amd as la
    B, H = 2, 2
    x = _data(T, B, H, T, decay, bf16)
    dt = torch.bfloat16 if bf16 else torch.float32
    t = {n: torch.from_numpy(x[n]).to(DEV).to(torch.float32 if n in ("gk", "h0") else dt).requires_grad_(True) for n in NAMES + ("h0",)}
    o, h = la.dplr_delta_rule_recurrent(*(t[n] for n in NAMES), 0.125, t["h0"])
    o_ref, h_ref = od.dplr_delta_rule_recurrent(*(x[n] for n in NAMES), 0.125, x["h0"])
    tol = 2e-2 if bf16 else 1e-4
    assert max_rel(o.detach().float().cpu().numpy(), o_ref) < tol and max_rel(h.detach().cpu().numpy(), h_ref) < tol
    with torch.no_grad():
        o2, h2 = la.dplr_delta_rule_recurrent(*(t[n] for n in NAMES), 0.125, t["h0"])
    assert torch.equal(o2, o.detach()) and torch.equal(h2, h.detach())
    torch.autograd.backward([o, h], [torch.from_numpy(x["dO"]).to(DEV).to(dt), torch.from_numpy(x["dS"]).to(DEV)])
    ref = od.dplr_delta_rule_adjoint(*(x[n] for n in NAMES), x["dO"], x["dS"], 0.125, x["h0"])
    for n in NAMES + ("h0",):
        e = max_rel(t[n].grad.float().cpu().numpy(), ref["dS0" if n == "h0" else "d" + n])
        assert e < tol, (n, e)


def test_windows_of_chunks():
    import linearnexus_amd as la
    torch.manual_seed(1)
    B, H, T = 64, 32, 64 * 17 + 5
    r = lambda: torch.randn(B, H, T, 64, device=DEV)
    kk = torch.nn.functional.normalize(r(), dim=-1)
    t = [r().bfloat16(), r().bfloat16(), r().bfloat16(), (-kk).bfloat16(), (kk * torch.rand(B, H, T, 64, device=DEV)).bfloat16(), -0.6 * torch.rand(B, H, T, 64, device=DEV)]
    dO = r().bfloat16()

    def run(rows):
        x = [u[rows].detach().clone().requires_grad_(True) for u in t]
        o, h = la.dplr_delta_rule_recurrent(*x)
        with torch.no_grad():
            o2, h2 = la.dplr_delta_rule_recurrent(*x)
        return [o.detach(), h.detach(), o2, h2, *torch.autograd.grad(o, x, dO[rows])]

    full, part = run(slice(0, B)), run(slice(61, 62))
    for a, b in zip(full, part):
        assert torch.isfinite(b.float()).all() and torch.equal(a[61:62], b)
