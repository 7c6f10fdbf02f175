"""The two forms of the forward scan at dk <= 128 -- 64-column slabs with everything in the compute waves, 32-column slabs whose outputs
have waves of their own a chunk behind -- give the same bits, and a segmented prompt, whose first pass forms no outputs, what one chain gives."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(B, H, T, dk, dv, seed=5):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    rows = lambda: (rnd(B, H, T, dk) * dk ** -0.5).bfloat16()  # of length about one: stable also where nothing is normalised
    return (rows(), rows(), rnd(B, H, T, dv).bfloat16(),
            -0.1 * torch.rand(B, H, T, generator=gen, device=DEV), torch.rand(B, H, T, generator=gen, device=DEV))


def _run(monkeypatch, slab, x, grads, cu=None, l2norm=True):
    import linearnexus_amd as la
    from linearnexus_amd import linear_attn
    monkeypatch.setitem(linear_attn._test_hooks, "scan_slab", slab)
    x = [t.clone().requires_grad_(grads) for t in x]
    q, k, v, g, beta = x
    o, S = la.gated_delta_rule_chunkwise(q, k, v, g, beta, use_qk_l2norm=l2norm, cu_seqlens=cu)
    return [o, S] + (list(torch.autograd.grad((o.float() ** 2).sum() + S.sum(), x)) if grads else [])


@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("grads,l2norm", [(False, True), (True, True), (True, False)])
def test_slabs_agree(monkeypatch, dk, chunks, grads, l2norm):
    x = _inputs(2, 3, 64 * chunks - 5, dk, 128)
    for a, b in zip(_run(monkeypatch, 32, x, grads, l2norm=l2norm), _run(monkeypatch, 64, x, grads, l2norm=l2norm)):
        assert torch.equal(a, b)


def test_slabs_agree_packed(monkeypatch):
    """Sequences of no, one and several chunks side by side."""
    cu = torch.tensor([0, 0, 1, 64, 129, 129, 500, 700], dtype=torch.int32, device=DEV)
    x = _inputs(1, 2, 700, 128, 64)
    for a, b in zip(_run(monkeypatch, 32, x, True, cu), _run(monkeypatch, 64, x, True, cu)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("H,chunks", [(1, 5), (40, 7)])  # 32- and 64-column slabs in the first pass
@pytest.mark.parametrize("dk", [64, 128])
def test_final_states_alone(monkeypatch, dk, H, chunks):
    """Two segments: the first pass leaves their transitions.  The final state passes through one more product of fp32 accuracy; what differs is
    the rounding of the columns that start from the identity instead of the state, 2^-9 of a value at every product."""
    x = _inputs(1, H, 64 * chunks - 9, dk, 64)
    monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "1")
    with torch.no_grad():
        o1, S1 = _run(monkeypatch, 0, x, False)
        monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "2")
        o2, S2 = _run(monkeypatch, 0, x, False)
    for a, b in ((o1, o2), (S1, S2)):
        assert ((a - b).float().norm() / a.float().norm()).item() < 2e-2


@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("T", [1, 61, 64, 333])
@pytest.mark.parametrize("token_first", [False, True])
@pytest.mark.parametrize("gated", [False, True])
def test_output_forms(monkeypatch, dk, T, token_first, gated):
    """Outputs in fp32 are the bf16 ones widened, in both forms and both layouts."""
    from linearnexus_amd import linear_attn
    q, k, v, g, beta = (t.transpose(1, 2).contiguous().transpose(1, 2) if token_first and t.dim() == 4 else t for t in _inputs(2, 3, T, dk, 64))
    results = []
    for slab in (64, 32):
        monkeypatch.setitem(linear_attn._test_hooks, "scan_slab", slab)
        for dtype in (torch.bfloat16, torch.float32):
            with torch.no_grad():
                o, S = linear_attn._chunk(q, k, v, g if gated else None, beta, dk ** -0.5, None, 64, gated, dtype, False, None)
            assert o.dtype == dtype
            results.append((o.float(), S))
    for o, S in results[1:]:
        assert torch.equal(o, results[0][0]) and torch.equal(S, results[0][1])
