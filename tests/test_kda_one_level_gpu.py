"""bf16 per-channel gates whose chunk's whole decay fits one factor a token (LNX_KDA_NEAR, csrc/chunk_common.h: 80 in units of log 2, per set of 64
channels) take their pairs in one level in kda_prepare, others in a hierarchy of levels: both, the limit between them and calls that mix them, against the
fp64 oracle."""
import numpy as np
import pytest
import torch

from conftest import max_rel
from oracle import recurrent as rc
from oracle.adjoint import delta_rule_adjoint
from oracle.gate import kda_gate, kda_gate_grad
from oracle.inputs import make_inputs, to_bf16_grid

pytestmark = pytest.mark.gpu
DEV = "cuda"
LIMIT = 80 * np.log(2.0) / 64  # mean decay of a token at the limit, full chunk


def _gates(which, T, dk, rng):
    g = -rng.random((1, 2, T, dk)).astype(np.float32)
    whole = lambda scale: g / g.reshape(1, 2, -1, 64, dk).sum(3).repeat(64, 2).reshape(g.shape) * -64 * LIMIT * scale if T % 64 == 0 else g
    if which == "below":
        return whole(0.999)
    if which == "above":
        return whole(1.001)
    if which in ("first_channel", "one_channel"):  # of the second chunk, in the first or the last set: the others stay in one level
        g *= 0.1
        g[:, :, 64:128, 3 if which == "first_channel" else dk - 3] = -3.0
        return g
    if which == "one_token":
        g *= 0.1
        g[:, :, 70] = -200.0
        return g
    if which == "zero":
        return np.zeros_like(g)
    assert which == "ragged"
    return g * 0.3


@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("which,T", [("below", 128), ("above", 128), ("first_channel", 192), ("one_channel", 192), ("one_token", 192), ("zero", 128), ("ragged", 65), ("ragged", 33), ("ragged", 143)])
def test_forward_and_gradients(which, T, dk, l2):
    import linearnexus_amd as la
    x = make_inputs(7, 1, 2, T, dk, 64, gate="vector", with_state=True, with_grad=True, normalize=not l2)
    x["g"] = np.ascontiguousarray(_gates(which, T, dk, np.random.default_rng(1)), np.float32)
    for n in ("q", "k", "v", "dO"):
        x[n] = to_bf16_grid(x[n])
    leaves = {n: torch.from_numpy(x[n]).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32).requires_grad_(True) for n in ("q", "k", "v", "g", "beta", "S0")}
    o, S = la.kda_chunkwise(leaves["q"], leaves["k"], leaves["v"], leaves["g"], leaves["beta"], None, leaves["S0"], 64, l2)
    grads = torch.autograd.grad([o, S], list(leaves.values()), [torch.from_numpy(x["dO"]).to(DEV), torch.from_numpy(x["dS"]).to(DEV)])
    d = {n: a.astype(np.float64) for n, a in x.items()}
    ro, rS = rc.kda_recurrent(d["q"], d["k"], d["v"], d["g"], d["beta"], None, d["S0"], l2)
    ref = delta_rule_adjoint(x["q"], x["k"], x["v"], x["beta"], x["dO"], x["g"], x["dS"], None, x["S0"], l2)
    errs = {"o": max_rel(o.detach().cpu().numpy(), ro), "S": max_rel(S.detach().cpu().numpy(), rS)}
    errs.update({"d" + n: max_rel(t.float().cpu().numpy(), ref["d" + n]) for n, t in zip(leaves, grads)})
    assert all(e < 2e-2 for e in errs.values()), errs


@pytest.mark.parametrize("dk", [64, 128])
def test_limit_joins_its_two_sides(dk):
    """Gates 1e-5 on either side of the limit (the fp32 sums of 64 of them are within 4e-6) are the same gates to bf16: what differs is the way.
    Either is within 5e-3 of fp64 in every one of these (they differ by 1.1e-3 to 2.7e-3)."""
    import linearnexus_amd as la
    x = make_inputs(8, 1, 2, 128, dk, 64, gate="vector", with_grad=True)
    x["g"] = np.ascontiguousarray(_gates("below", 128, dk, np.random.default_rng(2)), np.float32) / np.float32(0.999)

    def run(scale):
        leaves = [torch.from_numpy((x[n] * np.float32(scale if n == "g" else 1)).astype(np.float32)).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32).requires_grad_(True)
                  for n in ("q", "k", "v", "g", "beta")]
        o, _ = la.kda_chunkwise(*leaves, use_qk_l2norm=False)
        return [o.detach(), *torch.autograd.grad(o, leaves, torch.from_numpy(x["dO"]).to(DEV))]

    low, high = run(1 - 1e-5), run(1 + 1e-5)
    assert not torch.equal(low[0], high[0])
    for a, b in zip(low, high):
        a, b = a.float(), b.float()
        assert (a - b).norm() < 1e-2 * b.norm()


@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("channel,T", [(3, 192), (-3, 192), (None, 65), (None, 143)])
def test_raw_gates(channel, T, dk, l2):
    """The limit sees the activated gate, and rows past the end, whose raw zeros would not activate to zero, are out of it."""
    import linearnexus_amd as la
    x = make_inputs(12, 1, 2, T, dk, 64, gate="vector", with_state=True, with_grad=True, normalize=not l2)
    raw = np.random.default_rng(2).standard_normal((1, 2, T, dk)).astype(np.float32) - 1
    if channel is not None:
        raw[:, :, 64:128, channel] = 30.0
    A = np.log(np.array([0.1, 0.2], np.float32))
    for n in ("q", "k", "v", "dO"):
        x[n] = to_bf16_grid(x[n])
    raw = to_bf16_grid(raw)
    flat = raw.transpose(0, 2, 1, 3).reshape(1, T, 2 * dk)
    x["g"] = kda_gate(flat, A, dk)[0].transpose(0, 2, 1, 3)
    bf = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV).bfloat16().requires_grad_(True)
    leaves = {"q": bf(x["q"]), "k": bf(x["k"]), "v": bf(x["v"]), "g": bf(raw), **{n: torch.from_numpy(x[n]).to(DEV).requires_grad_(True) for n in ("beta", "S0")}}
    o, S = la.kda_chunkwise_raw_gate(*(leaves[n] for n in ("q", "k", "v", "g", "beta")), torch.from_numpy(A).to(DEV), None, None, leaves["S0"], 64, l2)
    grads = torch.autograd.grad([o, S], list(leaves.values()), [torch.from_numpy(x["dO"]).to(DEV), torch.from_numpy(x["dS"]).to(DEV)])
    d = {n: a.astype(np.float64) for n, a in x.items()}
    ro, rS = rc.kda_recurrent(d["q"], d["k"], d["v"], d["g"], d["beta"], None, d["S0"], l2)
    ref = delta_rule_adjoint(x["q"], x["k"], x["v"], x["beta"], x["dO"], x["g"], x["dS"], None, x["S0"], l2)
    ref["dg"] = kda_gate_grad(flat, A, dk, ref["dg"].transpose(0, 2, 1, 3))[0].reshape(1, T, 2, dk).transpose(0, 2, 1, 3)
    errs = {"o": max_rel(o.detach().cpu().numpy(), ro), "S": max_rel(S.detach().cpu().numpy(), rS)}
    errs.update({"d" + n: max_rel(t.float().cpu().numpy(), ref["d" + n]) for n, t in zip(leaves, grads)})
    assert all(e < 2e-2 for e in errs.values()), errs


def test_gates_above_zero_and_nan_keep_the_levels():
    """A gate above zero is outside the domain (its decay reads as 1 between neighbours at the levels) and is not taken to 2^+40 powers either:
    finite results; NaN stays in its own head."""
    import linearnexus_amd as la
    x = make_inputs(9, 1, 2, 128, 64, 64, gate="vector", with_grad=True)
    x["g"][:, 0, 5, 3] = 1e-3
    leaves = [torch.from_numpy(x[n]).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32).requires_grad_(True) for n in ("q", "k", "v", "g", "beta")]
    o, _ = la.kda_chunkwise(*leaves, use_qk_l2norm=False)
    gr = torch.autograd.grad(o, leaves, torch.from_numpy(x["dO"]).to(DEV))
    assert all(torch.isfinite(t).all() for t in (o, *gr))
    x["g"][:, 1, 70, 3] = np.nan
    leaves = [torch.from_numpy(x[n]).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32).requires_grad_(True) for n in ("q", "k", "v", "g", "beta")]
    o2, _ = la.kda_chunkwise(*leaves, use_qk_l2norm=False)
    gr2 = torch.autograd.grad(o2, leaves, torch.from_numpy(x["dO"]).to(DEV))
    assert torch.equal(o2[:, 0], o[:, 0]) and torch.isnan(o2[:, 1, 70:]).any()
    assert all(torch.equal(a[:, 0], b[:, 0]) for a, b in zip(gr, gr2))


@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("size", [2.0 ** 100, 2.0 ** -100])
def test_sizes_at_the_ends_of_the_range(size, dk):
    """Rows near the ends of the range keep the levels, whose factors are none above one: o is linear in q, whatever the size of q."""
    import linearnexus_amd as la
    x = make_inputs(10, 1, 2, 128, dk, 64, gate="vector", with_state=True)
    x["g"] = np.ascontiguousarray(_gates("below", 128, dk, np.random.default_rng(3)), np.float32)
    t = {n: torch.from_numpy(a).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32) for n, a in x.items()}
    run = lambda q: la.kda_chunkwise(q, t["k"], t["v"], t["g"], t["beta"], None, t["S0"], 64, False)[0].double()
    want, got = run(t["q"]), run(t["q"] * size) / size
    assert (got - want).norm() < 2e-2 * want.norm()  # each within 1e-2 of the same values


@pytest.mark.parametrize("dk", [64, 128])
def test_one_key_beyond_a_factor(dk):
    """A key of 2^100 in one channel of one late token of a chunk, queries of 2^-100 in that channel: their products are ordinary numbers."""
    import linearnexus_amd as la
    x = make_inputs(11, 1, 2, 128, dk, 64, gate="vector", with_state=True)
    x["g"] = np.ascontiguousarray(_gates("below", 128, dk, np.random.default_rng(4)), np.float32)
    x["k"][..., 7], x["S0"][..., 7, :] = 0.0, 0.0
    x["k"][:, :, 60, 7] = 2.0 ** 100
    x["q"][..., 7] *= 2.0 ** -100
    for n in "qkv":
        x[n] = to_bf16_grid(x[n])
    x["beta"][:, :, 60] = 0.5
    t = {n: torch.from_numpy(a).to(DEV).to(torch.bfloat16 if n in "qkv" else torch.float32) for n, a in x.items()}
    o, _ = la.kda_chunkwise(t["q"], t["k"], t["v"], t["g"], t["beta"], None, t["S0"], 64, False)
    d = {n: a.astype(np.float64) for n, a in x.items()}
    ro, _ = rc.kda_recurrent(d["q"], d["k"], d["v"], d["g"], d["beta"], None, d["S0"], False)
    assert max_rel(o.cpu().numpy(), ro) < 2e-2


@pytest.mark.parametrize("t", [1, 37, 63])
def test_an_infinite_query_is_infinite(t):
    """Positive values all along the one channel that the infinite query reads: the sum is +inf, and only in that token's row."""
    import linearnexus_amd as la
    gen = torch.Generator(device=DEV).manual_seed(t)
    T, D, c = 64, 64, 5
    q, k = torch.randn(1, 1, T, D, device=DEV, generator=gen), torch.zeros(1, 1, T, D, device=DEV)
    k[..., c] = 0.1 + 0.1 * torch.rand(1, 1, T, device=DEV, generator=gen)
    q[0, 0, t] = 0.0
    q[0, 0, t, c] = float("inf")
    v = 1 + torch.rand(1, 1, T, D, device=DEV, generator=gen)
    S0 = torch.zeros(1, 1, D, D, device=DEV)
    S0[:, :, c] = 0.5
    o, _ = la.kda_chunkwise(q.bfloat16(), k.bfloat16(), v.bfloat16(), torch.full((1, 1, T, D), -0.02, device=DEV), torch.full((1, 1, T), 0.1, device=DEV), None, S0, 64, False)
    others = torch.arange(T, device=DEV) != t
    assert torch.isfinite(o[:, :, others]).all() and (o[0, 0, t] == float("inf")).all()
