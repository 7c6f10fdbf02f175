"""The RWKV-7 scan where a document ends inside a row: the op has no cu_seqlens, a caller without it wipes the state with a large
negative gate.  Everything after the reset has to be as exact as without it, and the reset itself down to -inf must not leave a
NaN: outputs, final state and gradients against the fp64 oracle and its adjoint, fp32, resets of all channels and of some, at the
edges of the kernels' blocks of 16 tokens and chunks of 64, one after the other and in a row that ends inside a block.

The bound: at most 200 tokens of fp32 sums of 64 products.  Each rounds to 6e-8 of its largest term, a gradient passes about ten
sums in a row, and the largest element sits within a factor of 5 of what a sum's terms reach: 10 * 5 * 6e-8 = 3e-6 of max|ref|, doubled."""
import numpy as np
import pytest
import torch

from oracle import dplr as od
from conftest import max_rel

DEV = "cuda"
NAMES = ("q", "k", "v", "a", "b", "gk")
LOWEST = float(np.finfo(np.float32).min)
BOUND = 6e-6
D = 64


def _data(seed, B, H, T):
    r = np.random.default_rng(seed)
    n = lambda *s: r.standard_normal(s).astype(np.float32)
    kk = n(B, H, T, D)
    kk /= np.linalg.norm(kk, axis=-1, keepdims=True)
    return dict(q=n(B, H, T, D), k=n(B, H, T, D), v=n(B, H, T, D), a=-kk, b=kk * r.random((B, H, T, D)).astype(np.float32),
                gk=-0.6065 * r.random((B, H, T, D)).astype(np.float32), h0=n(B, H, D, D) * 0.5, dO=n(B, H, T, D), dS=n(B, H, D, D) * 0.3)


def _check(x):
    import linearnexus_amd as la
    t = {n: torch.from_numpy(x[n]).to(DEV).requires_grad_(True) for n in NAMES + ("h0",)}
    o, h = la.dplr_delta_rule_recurrent(*(t[n] for n in NAMES), 0.125, t["h0"])
    o_ref, h_ref = od.dplr_delta_rule_recurrent(*(x[n] for n in NAMES), 0.125, x["h0"])
    g = torch.autograd.grad([o, h], [t[n] for n in NAMES + ("h0",)], [torch.from_numpy(x["dO"]).to(DEV), torch.from_numpy(x["dS"]).to(DEV)])
    ref = od.dplr_delta_rule_adjoint(*(x[n] for n in NAMES), x["dO"], x["dS"], 0.125, x["h0"])
    err = {"o": max_rel(o.detach().cpu().numpy(), o_ref), "h": max_rel(h.detach().cpu().numpy(), h_ref)}
    for n, u in zip(NAMES + ("h0",), g):
        err["d" + n] = max_rel(u.cpu().numpy(), ref["dS0" if n == "h0" else "d" + n])
    print({n: f"{e:.1e}" for n, e in err.items()})
    assert all(e < BOUND for e in err.values()), err  # NaN fails, too


@pytest.mark.gpu
@pytest.mark.parametrize("gate", [-1e3, -1e4, -1e9, LOWEST, -np.inf])
@pytest.mark.parametrize("tokens", [(0,), (63,), (64,), (80,), (95, 96, 97), (5, 70, 199)])
def test_reset_of_every_channel(gate, tokens):
    x = _data(len(tokens) + tokens[0], 1, 2, 200)
    x["gk"][:, :, list(tokens)] = gate
    _check(x)


@pytest.mark.gpu
@pytest.mark.parametrize("gate", [-1e4, LOWEST, -np.inf])
def test_reset_of_some_channels(gate):
    x = _data(7, 2, 2, 150)
    x["gk"][:, 0, 37, ::17] = gate      # some channels of one head
    x["gk"][1, :, 64:70, 3] = gate      # one channel, six tokens in a row
    _check(x)


@pytest.mark.gpu
@pytest.mark.parametrize("gate", [-2.0, -6.0, -30.0])
def test_strong_decay_of_some_blocks(gate):
    """Blocks whose decays leave the range that one reference token can span, next to blocks that do not."""
    x = _data(11, 1, 2, 130)
    x["gk"][:, :, 16:48] += gate
    x["gk"][:, :, 100:, ::9] += gate
    _check(x)


@pytest.mark.gpu
def test_nan_gate_stays_visible():
    import linearnexus_amd as la
    x = {n: torch.from_numpy(a).to(DEV) for n, a in _data(3, 1, 1, 128).items()}
    x["gk"][0, 0, 70, 5] = float("nan")
    o, h = la.dplr_delta_rule_recurrent(*(x[n] for n in NAMES), 0.125, x["h0"])
    assert torch.isfinite(o[:, :, :64]).all() and torch.isnan(o[:, :, 70:]).all() and torch.isnan(h[0, 0, 5]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("decay", [0.0, 0.01, 1.0])
@pytest.mark.parametrize("reset", [None, -np.inf])
def test_relative_error(decay, reset):
    """RWKV-7's decays, weaker ones and none over eight chunks, in the 2-norm: 1e-6.  The kernels' sums have 64 terms of one chain at most
    (sqrt(64 / 2) * 3.4e-8 = 1.9e-7 of the sum); without decay a state carries the error of eight chunks, sqrt(8) * 1.9e-7 = 5.4e-7, and
    a gradient that of two such sums."""
    import linearnexus_amd as la
    x = _data(21, 1, 2, 512)
    x["gk"] *= np.float32(decay)
    if reset is not None:
        x["gk"][:, :, [80, 333]] = reset
    t = {n: torch.from_numpy(x[n]).to(DEV).requires_grad_(True) for n in NAMES + ("h0",)}
    o, h = la.dplr_delta_rule_recurrent(*(t[n] for n in NAMES), 0.125, t["h0"])
    g = torch.autograd.grad([o, h], [t[n] for n in NAMES + ("h0",)], [torch.from_numpy(x["dO"]).to(DEV), torch.from_numpy(x["dS"]).to(DEV)])
    o_ref, h_ref = od.dplr_delta_rule_recurrent(*(x[n] for n in NAMES), 0.125, x["h0"])
    ref = od.dplr_delta_rule_adjoint(*(x[n] for n in NAMES), x["dO"], x["dS"], 0.125, x["h0"])
    pairs = [("o", o, o_ref), ("h", h, h_ref)] + [("d" + n, u, ref["dS0" if n == "h0" else "d" + n]) for n, u in zip(NAMES + ("h0",), g)]
    err = {n: float(np.linalg.norm(u.detach().cpu().numpy() - r) / np.linalg.norm(r)) for n, u, r in pairs}
    print({n: f"{e:.1e}" for n, e in err.items()})
    assert all(e < 1e-6 for e in err.values()), err


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("decay", [4.0, 10.0])
def test_gate_gradient_behind_strong_decays(decay, dtype):
    """What flows through a strong decay is small next to what a token gives its own output: the gates' gradients must not carry the
    rounding of that, 2-norm, fp32 gates and their gradients in both types.  A block's sums have at most 16 terms of the flow's size on
    each side, every one rounded in a product of 64 terms (1.9e-7 of itself): sqrt(2 * 16) * 1.9e-7 = 1.1e-6 if all were as large as the
    sum; the mean of the token's place in the block halves their number, 7.5e-7."""
    import linearnexus_amd as la
    x = _data(22, 1, 2, 300)
    x["gk"] *= np.float32(decay)
    t = {n: torch.from_numpy(x[n]).to(DEV).to(dtype if n in NAMES[:5] else torch.float32).requires_grad_(True) for n in NAMES + ("h0",)}
    y = {n: u.detach().float().cpu().numpy() for n, u in t.items()}
    o, h = la.dplr_delta_rule_recurrent(*(t[n] for n in NAMES), 0.125, t["h0"])
    d_o = torch.from_numpy(x["dO"]).to(DEV).to(dtype)
    dgk, = torch.autograd.grad([o, h], [t["gk"]], [d_o, torch.from_numpy(x["dS"]).to(DEV)])
    ref = od.dplr_delta_rule_adjoint(*(y[n] for n in NAMES), d_o.float().cpu().numpy(), x["dS"], 0.125, y["h0"])["dgk"]
    err = float(np.linalg.norm(dgk.cpu().numpy() - ref) / np.linalg.norm(ref))
    print(f"{err:.1e}")
    assert err < 7.5e-7, err
