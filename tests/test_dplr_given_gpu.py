"""Products of the RWKV-7 chunk kernels with v and dO: bf16 tensors go through bf16 products of the other operand's parts, fp32 ones
through fp32 products.  The same values in both types give the same sums in another order."""
import numpy as np
import pytest
import torch
from oracle.inputs import to_bf16_grid

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAMES = ("q", "k", "v", "a", "b", "gk")


@pytest.mark.parametrize("size", [1.0, 2.0 ** 40, 2.0 ** -40])
@pytest.mark.parametrize("T,decay", [(16, 1.0), (63, 1.0), (64, 10.0), (65, 0.0), (330, 1.0)])
def test_types_agree(T, decay, size):
    """v and dO of any size lose nothing.  Either type's sums are within sqrt(8) * 1.9e-7 of the exact ones over these lengths (64 terms a
    chain, up to eight chunks of them), the gates' gradients within 7.5e-7 (sums over a block's tokens of such): twice that apart."""
    import linearnexus_amd as la
    r = np.random.default_rng(T)
    n = lambda *s: r.standard_normal(s).astype(np.float32)
    B, H, D = 1, 3, 64
    kk = n(B, H, T, D)
    kk /= np.linalg.norm(kk, axis=-1, keepdims=True)
    x = dict(q=n(B, H, T, D), k=n(B, H, T, D), v=n(B, H, T, D) * size, a=-kk, b=kk * r.random((B, H, T, D)), gk=-0.6065 * decay * r.random((B, H, T, D)))
    x = {m: torch.from_numpy((to_bf16_grid(u.astype(np.float32)) if m != "gk" else u).astype(np.float32)).to(DEV) for m, u in x.items()}
    h0 = torch.from_numpy(n(B, H, D, D) * np.float32(size)).to(DEV)
    d_o, dS = torch.from_numpy(to_bf16_grid(n(B, H, T, D))).to(DEV), torch.from_numpy(n(B, H, D, D)).to(DEV)

    def run(dt):
        t = {m: (u.clone() if m == "gk" else u.to(dt)).requires_grad_(True) for m, u in x.items()}
        s0 = h0.clone().requires_grad_(True)
        o, h = la.dplr_delta_rule_recurrent(*(t[m] for m in NAMES), 0.125, s0)
        dgk, ds0, dv = torch.autograd.grad([o, h], [t["gk"], s0, t["v"]], [d_o.to(dt), dS])
        return {"o": o, "h": h, "dh0": ds0, "dgk": dgk, "dv": dv}

    low, full = run(torch.bfloat16), run(torch.float32)
    for m, want in full.items():
        got = low[m].detach().double()
        want = want.detach().double()
        err = float((got - want).norm() / want.norm())
        bound = 2 ** -9 if low[m].dtype == torch.bfloat16 else 1.5e-6 if m == "dgk" else 1.1e-6
        assert err < bound, (m, err)
