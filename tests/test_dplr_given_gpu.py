"""Products of the RWKV-7 chunk kernels with v and dO: bf16 tensors go through bf16 products of the other operand's parts, fp32 ones
through fp32 products.  The same values in both types give the same sums in another order."""
import numpy as np
import pytest
import torch
from oracle.dplr import dplr_delta_rule_recurrent
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


@pytest.mark.parametrize("decay", [1.0, 3.0, 4.0, 10.0])
def test_final_state_is_as_exact_as_from_fp32_tensors(decay):
    """However few tokens the gates leave to the state's sums.  The two errors are each the norm over 16384 roundings, 0.8 % from seed to seed."""
    import linearnexus_amd as la
    r = np.random.default_rng(5)
    n = lambda *s: r.standard_normal(s).astype(np.float32)
    B, H, T, D = 1, 4, 512, 64
    kk = n(B, H, T, D)
    kk /= np.linalg.norm(kk, axis=-1, keepdims=True)
    x = dict(q=n(B, H, T, D), k=n(B, H, T, D), v=n(B, H, T, D), a=-kk, b=kk * r.random((B, H, T, D)))
    x = {m: to_bf16_grid(u.astype(np.float32)) for m, u in x.items()}
    x["gk"], h0 = (-0.606531 * decay / (1 + np.exp(-n(B, H, T, D)))).astype(np.float32), n(B, H, D, D)
    want = dplr_delta_rule_recurrent(*(x[m].astype(np.float64) for m in NAMES), 0.125, h0.astype(np.float64))[1]

    def error(dt):
        _, h = la.dplr_delta_rule_recurrent(*(torch.from_numpy(x[m]).to(DEV).to(torch.float32 if m == "gk" else dt) for m in NAMES), 0.125, torch.from_numpy(h0).to(DEV))
        return np.linalg.norm(h.double().cpu().numpy() - want) / np.linalg.norm(want)

    low, full = error(torch.bfloat16), error(torch.float32)
    assert low < 1.03 * full and full < 1e-7, (low, full)


def classes(x):
    """0 finite, 1 and 2 the infinities, 3 NaN"""
    return torch.where(x.isnan(), 3, torch.where(x.isinf(), torch.where(x > 0, 1, 2), 0))


@pytest.mark.parametrize("T", [64, 150])
@pytest.mark.parametrize("what", ["pair", "d_o", "v", "nan"])
def test_infinite_values(what, T):
    """What is not finite is so at the same places in either type: a pair's product <q, k> beyond the fp32 range (in a channel that a and b do
    not touch), infinities in dO of the first chunk and in v, NaN in v.  Every term of a sum has one sign or is NaN in both, so the class of a sum
    does not hang on its order."""
    import linearnexus_amd as la
    r = np.random.default_rng(T)
    n = lambda *s: torch.from_numpy(to_bf16_grid(r.standard_normal(s).astype(np.float32)).astype(np.float32)).to(DEV)
    B, H, D = 1, 2, 64
    kk = torch.nn.functional.normalize(n(B, H, T, D), dim=-1)
    x = dict(q=n(B, H, T, D), k=n(B, H, T, D), v=n(B, H, T, D), a=-kk, b=kk * torch.sigmoid(n(B, H, T, D)))
    x = {m: u.bfloat16().float() for m, u in x.items()}
    gk, h0, d_o, dS = -0.6065 * torch.sigmoid(n(B, H, T, D)), n(B, H, D, D), n(B, H, T, D), n(B, H, D, D)
    inf = float("inf")
    if what == "pair":
        x["a"][..., 7] = x["b"][..., 7] = 0
        x["q"][0, 0, 37, 7], x["k"][0, 0, 21, 7], x["k"][0, 0, 3, 7] = 2.0 ** 80, 2.0 ** 75, -2.0 ** 35
    elif what == "d_o":
        d_o[0, 0, 40, 5], d_o[0, 0, 9, 11] = inf, -inf
    elif what == "v":
        x["v"][0, 0, 30, 5], x["v"][0, 0, T - 1, 9] = -inf, inf
    else:
        x["v"][0, 0, 30, 5] = float("nan")

    def run(dt):
        t = {m: u.to(dt).requires_grad_(True) for m, u in x.items()}
        t["gk"], s0 = gk.clone().requires_grad_(True), h0.clone().requires_grad_(True)
        o, h = la.dplr_delta_rule_recurrent(*(t[m] for m in NAMES), 0.125, s0)
        grads = torch.autograd.grad([o, h], [*(t[m] for m in NAMES), s0], [d_o.to(dt), dS])
        return dict(zip(("o", "h", *("d" + m for m in NAMES), "dh0"), (o, h, *grads)))

    low, full = run(torch.bfloat16), run(torch.float32)
    reached = 0
    for m, want in full.items():
        want, got = classes(want.detach()), classes(low[m].detach())
        differ = (want != got).nonzero()
        assert len(differ) == 0, (m, len(differ), differ[:4].tolist(), want[tuple(differ[0])].item(), got[tuple(differ[0])].item())
        reached += int(((want > 0) & (want < 3)).sum() if what in ("pair", "d_o") else (want > 0).sum())
        # another head's row has none of it
        assert int((got[:, 1] > 0).sum()) == 0, m
    assert reached > 0
