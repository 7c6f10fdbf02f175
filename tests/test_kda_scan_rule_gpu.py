"""bf16 per-channel gates, dk = 128: few slabs run the chain in registers while the call fits the cache (2100 chunks of dv = 128, launch_fwd in
csrc/chunk_fwd.hip), else the one through LDS.  On either side of the line the library's choice gives the bits of the form that it should take, with
states saved and without, and the other form the same but for the order of fp32 sums: a rounding to bf16 moved by one step, 2^-8 of a value, here and there."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dv,H,chunks,slab", [(128, 5, 420, 32), (128, 6, 350, 32), (128, 6, 351, 64), (128, 1, 2101, 64), (64, 10, 280, 32), (64, 10, 281, 64), (256, 4, 350, 32), (256, 4, 351, 64)])
def test_choice(monkeypatch, dv, H, chunks, slab):
    import linearnexus_amd as la
    from linearnexus_amd import linear_attn
    monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "1")
    gen = torch.Generator(device=DEV).manual_seed(chunks)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    T = 64 * chunks - 5
    x = [(rnd(1, H, T, 128) * 128 ** -0.5).bfloat16(), (rnd(1, H, T, 128) * 128 ** -0.5).bfloat16(), rnd(1, H, T, dv).bfloat16(),
         -0.3 * torch.rand(1, H, T, 128, device=DEV, generator=gen), torch.rand(1, H, T, device=DEV, generator=gen)]

    def run(s, grad):
        monkeypatch.setitem(linear_attn._test_hooks, "scan_slab", s)
        with torch.set_grad_enabled(grad):
            o, S = la.kda_chunkwise(*(t.detach().requires_grad_(grad) for t in x))
        return o.detach(), S.detach()

    want = run(slab, False)
    for grad in (False, True):
        got = run(0, grad)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    for a, b in zip(run(96 - slab, False), want):
        assert torch.isfinite(a).all() and float((a.double() - b.double()).norm() / b.double().norm()) < 2 ** -8
