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
    """Slow decay, so that a segment's entering state matters to its end; the fp32 chain is the yardstick of both."""
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
        assert rel(b, t) <= (1e-5 if dtype == torch.float32 else 1.25 * rel(a, t) + 1e-3)
