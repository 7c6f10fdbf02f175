"""The dk = 256 scans (csrc/chunk_wide.hip) at every slab width -- 128 columns where there are that many chains, 64 and 32 -- give
the same bits: outputs, final state and gradients, lengths around the chunk, with and without a gate and an initial state.
(The 64- and 32-column slabs are compared with the oracle in test_dk256_gpu.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("T,with_state", [(1, True), (63, False), (64, True), (130, True)])
@pytest.mark.parametrize("B,H,dv,o_dtype", [(13, 16, 128, torch.bfloat16), (2, 2, 192, torch.bfloat16), (13, 16, 128, torch.float32)])
def test_slab_widths_agree(gate, T, with_state, B, H, dv, o_dtype, monkeypatch):
    from linearnexus_amd import linear_attn as m
    torch.manual_seed(T)
    r = lambda *s: torch.randn(*s, device=DEV)
    unit = lambda *s: torch.nn.functional.normalize(r(*s), dim=-1).bfloat16()
    x = [unit(B, H, T, 256), unit(B, H, T, 256), r(B, H, T, dv).bfloat16(), -0.1 * torch.rand(B, H, T, device=DEV) if gate else None,
         torch.rand(B, H, T, device=DEV), r(B, H, 256, dv) * 0.1 if with_state else None]
    do, dS = r(B, H, T, dv).to(o_dtype), r(B, H, 256, dv) * 0.1

    def run(slab):
        monkeypatch.setitem(m._test_hooks, "scan_slab", slab)
        t = [None if u is None else u.clone().requires_grad_(True) for u in x]
        q, k, v, g, beta, s0 = t
        o, S = m._chunk_forward(q, k, v, g, beta, s0, 256 ** -0.5, False, o_dtype, None, forward_only=False)
        o2, S2 = m._chunk_forward(*(None if u is None else u.detach() for u in (q, k, v, g, beta, s0)), 256 ** -0.5, False, o_dtype, None, forward_only=True)
        assert torch.equal(o, o2) and torch.equal(S, S2)
        return [o.detach(), S.detach(), *torch.autograd.grad([o, S], [u for u in t if u is not None], [do, dS])]

    auto, wide, narrow = run(0), run(64), run(32)
    for a, b, c in zip(auto, wide, narrow):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b) and torch.equal(a, c)
