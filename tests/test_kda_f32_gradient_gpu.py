"""An output gradient in fp32 (the per-channel gate's rule returns fp32 by default) is rounded to bf16 by the reverse scan as it reads it: the
gradients are bit for bit those of the rounded gradient."""
import pytest
import torch

DEV = "cuda"


def test_refused_where_the_query_says_no():
    from linearnexus_amd import _lib
    lib = _lib.load()
    a = _lib.ScanArgs(B=1, H=1, T=64, dk=64, dv=64, chunk=64, dtype=_lib.LNX_BF16, o_dtype=_lib.LNX_F32, gate=_lib.GATE_VECTOR)
    for dtype, dk, gate in ((_lib.LNX_BF16, 64, _lib.GATE_VECTOR), (_lib.LNX_BF16, 128, _lib.GATE_VECTOR), (_lib.LNX_BF16, 256, _lib.GATE_VECTOR),
                            (_lib.LNX_F32, 64, _lib.GATE_VECTOR), (_lib.LNX_BF16, 128, _lib.GATE_SCALAR), (_lib.LNX_BF16, 128, _lib.GATE_NONE)):
        a.dtype, a.dk, a.gate = dtype, dk, gate
        takes = dtype == _lib.LNX_BF16 and dk <= 128 and gate == _lib.GATE_VECTOR
        assert lib.lnx_chunk_rounds_d_o(a) == takes
        status = lib.lnx_chunk_bwd_d_o32(a, 16, None)  # the null tensors of `a` are refused before anything is read
        assert (status == -1 and b"required" in lib.lnx_last_error()) if takes else status != 0, lib.lnx_last_error()
    a.dtype, a.dk, a.gate = _lib.LNX_BF16, 128, _lib.GATE_VECTOR
    assert lib.lnx_chunk_bwd_d_o32(a, 20, None) == -2 and b"aligned" in lib.lnx_last_error()
    assert lib.lnx_chunk_bwd_d_o32(a, None, None) == -1 and lib.lnx_chunk_bwd_d_o32(None, 16, None) == -1 and lib.lnx_chunk_rounds_d_o(None) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dk,dv,slab", [(64, 64, 64), (64, 128, 64), (128, 64, 32), (128, 128, 64)])
@pytest.mark.parametrize("T,cu", [(1, None), (64, None), (65, None), (320, None), (330, [0, 0, 1, 64, 129, 330])])
@pytest.mark.parametrize("form", ["heads", "tokens", "expanded", "offset"])
def test_same_as_the_rounded_gradient(monkeypatch, dk, dv, slab, T, cu, form):
    import linearnexus_amd as la
    from linearnexus_amd import linear_attn
    monkeypatch.setitem(linear_attn._test_hooks, "scan_slab", slab)
    gen = torch.Generator(device=DEV).manual_seed(T + dk)
    B, H = (1 if cu else 2), 3
    n = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    tokens = form == "tokens"
    lay = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2) if tokens else t  # logical [B, H, T, d]
    x = [lay(n(B, H, T, dk) * dk ** -0.5).bfloat16(), lay(n(B, H, T, dk) * dk ** -0.5).bfloat16(), lay(n(B, H, T, dv)).bfloat16(), lay(-torch.rand(B, H, T, dk, device=DEV, generator=gen)),
         lay(torch.rand(B, H, T, device=DEV, generator=gen)), n(len(cu) - 1 if cu else B, H, dk, dv)]
    x = [t.requires_grad_(True) for t in x]
    d_o = lay(n(B, H, T, dv))
    if form == "expanded":
        d_o = n(B, H, 1, dv).expand(B, H, T, dv)
    if form == "offset":  # dense, but not on a 16-byte boundary
        d_o = torch.empty(B * H * T * dv + 1, device=DEV)[1:].view(B, H, T, dv).copy_(d_o)
    before = d_o.clone()
    offsets = None if cu is None else torch.tensor(cu, dtype=torch.int32, device=DEV)

    def grads(out, d):
        o, _ = la.kda_chunkwise(*x[:5], None, x[5], output_dtype=out, cu_seqlens=offsets)
        return torch.autograd.grad(o, x, d)

    for name, got, want in zip(("q", "k", "v", "g", "beta", "S0"), grads(torch.float32, d_o), grads(torch.bfloat16, d_o.bfloat16())):
        assert torch.isfinite(want).all() and torch.equal(got, want), name
    assert torch.equal(before, d_o)
