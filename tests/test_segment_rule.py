"""Which forward-only calls are cut into segments at dk <= 128, and that the calls next to the lines give what one chain gives."""
import pytest
import torch

from linearnexus_amd.linear_attn import _prefill_segments

DEV = "cuda"


@pytest.mark.parametrize("B,H,T,dv,dk,two_byte,vector,expected", [
    (1, 4, 4032, 128, 128, True, False, 1), (1, 4, 4033, 128, 128, True, False, 8), (1, 4, 16384, 128, 128, True, False, 16),
    (1, 6, 4096, 64, 64, True, False, 8), (1, 16, 8128, 128, 128, True, False, 1), (1, 16, 8192, 128, 128, True, False, 4),
    (2, 8, 32768, 128, 128, True, False, 8), (1, 17, 65536, 128, 128, True, False, 1), (1, 4, 8128, 128, 128, True, True, 1),
    (1, 8, 8192, 128, 128, True, True, 8), (1, 9, 65536, 128, 128, False, True, 1), (1, 8, 4096, 128, 128, False, False, 8),
])
def test_rule(monkeypatch, B, H, T, dv, dk, two_byte, vector, expected):
    monkeypatch.delenv("LNX_PREFILL_SEGMENTS", raising=False)
    assert _prefill_segments(B, H, T, dv, dk, two_byte, vector) == expected


@pytest.mark.gpu
@pytest.mark.parametrize("variant", ["delta", "gated", "kda"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,T,d,token_first", [(1, 4, 8193, 128, False), (2, 3, 4097, 64, False), (2, 2, 8200, 64, True), (1, 7, 8255, 128, True)])
def test_segments_against_one_chain(monkeypatch, variant, dtype, B, H, T, d, token_first):
    """Slow decay, so that a segment's entering state matters to its end; the fp32 chain is the yardstick of both.  The segments' states
    pass through one more product, in fp32: bf16 calls are within 1 % of the chain's error (measured: 0.3 %)."""
    import linearnexus_amd as la
    gen = torch.Generator(device=DEV).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    q, k = (torch.nn.functional.normalize(rnd(B, H, T, d), dim=-1).to(dtype) for _ in "qk")
    v, beta = rnd(B, H, T, d).to(dtype), torch.sigmoid(rnd(B, H, T))
    g = -torch.nn.functional.softplus(rnd(B, H, T, d) if variant == "kda" else rnd(B, H, T)) * 1e-3
    s0 = rnd(B, H, d, d)

    def run(nseg, cast):
        x = [t.to(cast) for t in (q, k, v)]
        if token_first:
            x = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in x]
        if nseg is None:
            monkeypatch.delenv("LNX_PREFILL_SEGMENTS", raising=False)
        else:
            monkeypatch.setenv("LNX_PREFILL_SEGMENTS", str(nseg))
        with torch.no_grad():
            if variant == "delta":
                return la.delta_rule_chunkwise(*x, beta, s0)
            return (la.kda_chunkwise if variant == "kda" else la.gated_delta_rule_chunkwise)(*x, g, beta, None, s0, 64, False)

    def rel(a, b):
        return float((a.double() - b.double()).norm() / b.double().norm())

    truth = run(1, torch.float32)
    chain, cut = run(1, dtype), run(None, dtype)
    for t, a, b in zip(truth, chain, cut):
        print(f"chain {rel(a, t):.2e} segments {rel(b, t):.2e}")
        assert rel(b, t) <= (2e-6 if dtype == torch.float32 else 1.01 * rel(a, t))


def _fp64(q, k, v, g, beta, s0, scale):
    """The chunked scan in 64 bits, scalar or no gate (mild decays: e^-G is formed)."""
    q, k, v, beta, S = (t.double() for t in (q, k, v, beta, s0))
    outs = []
    for t0 in range(0, q.shape[2], 64):
        Q, K, V, b = q[:, :, t0:t0 + 64] * scale, k[:, :, t0:t0 + 64], v[:, :, t0:t0 + 64], beta[:, :, t0:t0 + 64, None]
        G = torch.zeros_like(b) if g is None else torch.cumsum(g[:, :, t0:t0 + 64].double(), 2)[..., None]
        Kp, Km, Qp = K * G.exp(), (K * (-G).exp()).transpose(-1, -2).contiguous(), Q * G.exp()
        A = torch.tril(torch.matmul(Kp, Km), -1) * b
        D = torch.linalg.solve_triangular(torch.eye(b.shape[2], device=DEV, dtype=torch.float64) + A, b * (V - torch.matmul(Kp, S)), upper=False)
        outs.append(torch.matmul(Qp, S) + torch.matmul(torch.tril(torch.matmul(Qp, Km)), D))
        S = S * G[:, :, -1:].exp() + torch.matmul((K * (G[:, :, -1:] - G).exp()).transpose(-1, -2).contiguous(), D)
    return torch.cat(outs, 2), S


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,T,d,decay", [(4, 8192, 128, None), (8, 16384, 64, None), (4, 8192, 128, 0.1), (4, 8192, 128, 1e-3), (16, 8192, 128, None)])
def test_segments_are_as_exact_as_one_chain(monkeypatch, dtype, H, T, d, decay):
    """Against 64 bits, with decays down to none, where an error lives longest.  The chain's own error from run to run of the data spreads
    by 0.5 %; the segments' was at most 1.5 % above it (fp32, no gate: one more fp32 product of states)."""
    import linearnexus_amd as la
    gen = torch.Generator(device=DEV).manual_seed(T + H)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    q, k = (torch.nn.functional.normalize(rnd(1, H, T, d), dim=-1).to(dtype) for _ in "qk")
    v, beta, s0 = rnd(1, H, T, d).to(dtype), torch.sigmoid(rnd(1, H, T)), rnd(1, H, d, d) * 0.02
    g = None if decay is None else -torch.nn.functional.softplus(rnd(1, H, T)) * decay
    truth = _fp64(q, k, v, g, beta, s0, d ** -0.5)

    def errors(nseg):
        monkeypatch.delenv("LNX_PREFILL_SEGMENTS", raising=False)
        if nseg:
            monkeypatch.setenv("LNX_PREFILL_SEGMENTS", str(nseg))
        with torch.no_grad():
            out = la.delta_rule_chunkwise(q, k, v, beta, s0) if g is None else la.gated_delta_rule_chunkwise(q, k, v, g, beta, None, s0, 64, False)
        return [float((a.double() - t).norm() / t.norm()) for a, t in zip(out, truth)]

    chain, cut = errors(1), errors(None)
    print(f"chain o {chain[0]:.3e} S {chain[1]:.3e}, segments o {cut[0]:.3e} S {cut[1]:.3e}")
    assert all(b <= 1.03 * a for a, b in zip(chain, cut))
