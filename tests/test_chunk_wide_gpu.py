"""The dk = 256 scans (csrc/chunk_wide.hip) at every slab width -- 128 columns where there are that many chains, 64 and 32 -- give
the same bits: outputs, final state and gradients, lengths around the chunk, with and without a gate and an initial state.  That alone
compares the kernel with itself: rows of the 128-column slabs are compared with the oracle below, and the narrower ones in
test_dk256_gpu.py."""
import numpy as np
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


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("T", [64, 130])
def test_wide_slabs_against_the_oracle(gate, T):
    """208 chains, which take 128-column slabs by the library's own choice; three of them against fp64 at the bound of 2-byte inputs."""
    from conftest import max_rel
    from linearnexus_amd import linear_attn as m
    from oracle import recurrent as rc
    from oracle.adjoint import delta_rule_adjoint
    torch.manual_seed(T)
    B, H, dk, dv = 13, 16, 256, 128
    r = lambda *s: torch.randn(*s, device=DEV)
    unit = lambda *s: torch.nn.functional.normalize(r(*s), dim=-1).bfloat16()
    x = dict(q=unit(B, H, T, dk), k=unit(B, H, T, dk), v=r(B, H, T, dv).bfloat16(), beta=torch.rand(B, H, T, device=DEV), s0=r(B, H, dk, dv) * 0.1)
    if gate:
        x["g"] = -0.1 * torch.rand(B, H, T, device=DEV)
    do, dS = r(B, H, T, dv).bfloat16(), r(B, H, dk, dv) * 0.1
    t = {n: u.clone().requires_grad_(True) for n, u in x.items()}
    o, S = m._chunk_forward(t["q"], t["k"], t["v"], t.get("g"), t["beta"], t["s0"], dk ** -0.5, False, torch.bfloat16, None, forward_only=False)
    got = dict(zip(t, torch.autograd.grad([o, S], list(t.values()), [do, dS])))
    for b, h in ((0, 0), (6, 9), (12, 15)):
        c = lambda u: u.detach()[b:b + 1, h:h + 1].float().cpu().numpy().astype(np.float64)
        y = {n: c(u) for n, u in x.items()}
        if gate:
            o_ref, S_ref = rc.gated_delta_rule_recurrent(y["q"], y["k"], y["v"], y["g"], y["beta"], None, y["s0"], False)
        else:
            o_ref, S_ref = rc.delta_rule_recurrent(y["q"], y["k"], y["v"], y["beta"], y["s0"])
        ref = delta_rule_adjoint(y["q"], y["k"], y["v"], y["beta"], c(do), y.get("g"), c(dS), None, y["s0"], False)
        err = {"o": max_rel(c(o), o_ref), "S": max_rel(c(S), S_ref), **{n: max_rel(c(got[n]), ref["dS0" if n == "s0" else "d" + n]) for n in got}}
        assert all(e < 2e-2 for e in err.values()), (b, h, err)


@pytest.mark.parametrize("T,cu", [(1, None), (64, None), (129, None), (250, None), (330, None),
                                  (500, [0, 0, 1, 64, 129, 129, 130, 131, 200, 264, 265, 270, 300, 500])])
@pytest.mark.parametrize("gate", [False, True])
def test_normalised_rows_at_every_width(gate, T, cu, monkeypatch):
    """Rows normalised inside the kernels, where the narrow slabs' movers hold two chunks: no, one, even and odd numbers of chunks."""
    from linearnexus_amd import linear_attn as m
    B, H, dv = (1 if cu else 13), 16, 128
    torch.manual_seed(T)
    r = lambda *s: torch.randn(*s, device=DEV)
    x = [r(B, H, T, 256).bfloat16(), r(B, H, T, 256).bfloat16(), r(B, H, T, dv).bfloat16(), -0.1 * torch.rand(B, H, T, device=DEV) if gate else None,
         torch.rand(B, H, T, device=DEV)]
    do, dS = r(B, H, T, dv).bfloat16(), r(13, H, 256, dv) * 0.1
    cu = None if cu is None else torch.tensor(cu, dtype=torch.int32, device=DEV)

    def run(slab):
        monkeypatch.setitem(m._test_hooks, "scan_slab", slab)
        t = [None if u is None else u.clone().requires_grad_(True) for u in x]
        o, S = m._chunk_forward(*t, None, 256 ** -0.5, True, torch.bfloat16, cu, forward_only=False)[:2]
        o2, S2 = m._chunk_forward(*x, None, 256 ** -0.5, True, torch.bfloat16, cu, forward_only=True)[:2]
        assert torch.equal(o, o2) and torch.equal(S, S2)
        return [o.detach(), S.detach(), *torch.autograd.grad([o, S], [u for u in t if u is not None], [do, dS])]

    auto, wide, narrow = run(0), run(64), run(32)
    for a, b, c in zip(auto, wide, narrow):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b) and torch.equal(a, c)
