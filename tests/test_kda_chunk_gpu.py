"""The gradient kernel of the per-channel gate (csrc/chunk_kda.hip) and the L2 normalisation inside its kernels: value dimensions whose slabs fill
the ring of slab buffers exactly, unevenly and several times over, lengths around the chunk, packed batches with an empty sequence.  Bound 2e-2
of the largest value against the fp64 oracles (bf16 inputs, fp32 accumulation)."""
import numpy as np
import pytest
import torch

from conftest import max_rel
from linearnexus_amd import _lib
from oracle.adjoint import delta_rule_adjoint
from oracle.inputs import make_inputs
from test_chunk_bwd_gpu import _prep, check, gpu_grads
from test_chunk_fwd_gpu import gpu_chunk_fwd, oracle_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("dk,dv", [(128, 64), (128, 128), (128, 320), (64, 64), (64, 128), (64, 320)])
@pytest.mark.parametrize("T,cu", [(1, None), (64, None), (130, None), (200, [0, 3, 3, 67, 200])])
def test_gradients(dk, dv, T, cu, l2):
    B, H = (1 if cu else 2), 2
    x = make_inputs(93, B, H, T, dk, dv, gate="vector", with_state=not cu, with_grad=True, normalize=not l2)
    rng = np.random.default_rng(94)
    if l2:
        for n in "qk":
            x[n] = x[n] * np.exp(rng.standard_normal((B, H, T, 1))).astype(np.float32)
        a = _lib.ScanArgs(B=B, H=H, T=T, dk=dk, dv=dv, chunk=64, dtype=_lib.LNX_BF16, o_dtype=_lib.LNX_F32, gate=_lib.GATE_VECTOR)
        assert _lib.load().lnx_chunk_normalises_qk(a) == 1
    if cu:
        x["S0"], x["dS"] = ((rng.standard_normal((len(cu) - 1, H, dk, dv)) * s).astype(np.float32) for s in (0.02, 0.1))
    x, dt = _prep(x, True)
    if not cu:
        o_ref, S_ref = oracle_fwd(x, "vector", l2=l2)
        with torch.no_grad():
            o, S = gpu_chunk_fwd(x, "vector", dt, l2=l2)
        assert max_rel(o.float().cpu().numpy(), o_ref) < 2e-2 and max_rel(S.cpu().numpy(), S_ref) < 2e-2
    spans = [(i, lo, hi) for i, (lo, hi) in enumerate(zip(cu[:-1], cu[1:]))] if cu else [(0, 0, T)]
    parts = []
    for i, lo, hi in spans:
        dS, S0 = (x[n][i:i + 1] if cu else x[n] for n in ("dS", "S0"))
        if lo == hi:
            parts.append({"dS0": dS})
        else:
            parts.append(delta_rule_adjoint(*(x[n][:, :, lo:hi] for n in ("q", "k", "v", "beta", "dO", "g")), dS, None, S0, l2))
    ref = {n: np.concatenate([p[n] for p in parts if n in p], 2) for n in ("dq", "dk", "dv", "dbeta", "dg")}
    ref["dS0"] = np.concatenate([p["dS0"] for p in parts], 0)
    check(gpu_grads(x, "vector", dt, cu=None if cu is None else np.array(cu, np.int32), l2=l2), ref, 2e-2)


@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("H,T,cu", [(3, 500, None), (3, 64, None), (2, 700, [0, 0, 1, 64, 129, 129, 500, 700]), (56, 130, None), (60, 330, None)])
@pytest.mark.parametrize("f32_out", [False, True])
def test_forward_forms(monkeypatch, dk, H, T, cu, f32_out):
    """The chain in registers (32-column slabs) against the one through LDS (64-column slabs) and against the own choice, which at dk = 128 lies
    between 56 and 60 heads.  Both round the state and D to bf16 at the same places; what differs is the order of fp32 sums, which can move such
    a rounding by one step, 2^-8 of a value: 1e-2 of the largest."""
    import linearnexus_amd as la
    from linearnexus_amd import linear_attn
    gen = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x = [(rnd(1, H, T, dk) * dk ** -0.5).bfloat16(), (rnd(1, H, T, dk) * dk ** -0.5).bfloat16(), rnd(1, H, T, 128).bfloat16(),
         -0.3 * torch.rand(1, H, T, dk, generator=gen, device="cuda"), torch.rand(1, H, T, generator=gen, device="cuda")]
    out = torch.float32 if f32_out else torch.bfloat16
    monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "1")
    cu = None if cu is None else torch.tensor(cu, dtype=torch.int32, device="cuda")
    results = []
    for slab in (64, 32, 0):
        monkeypatch.setitem(linear_attn._test_hooks, "scan_slab", slab)
        y = [t.clone().requires_grad_() for t in x]
        with torch.no_grad():
            plain = la.kda_chunkwise(*y, cu_seqlens=cu, output_dtype=out)
        o, S = la.kda_chunkwise(*y, cu_seqlens=cu, output_dtype=out)
        assert torch.equal(plain[0], o) and torch.equal(plain[1], S)  # with and without saved states
        results.append([o, S, *torch.autograd.grad((o.float() ** 2).sum() + S.sum(), y)])
    for got in results[1:]:
        for a, b in zip(results[0], got):
            assert torch.isfinite(b).all() and max_rel(b.detach().float().cpu().numpy(), a.detach().float().cpu().numpy()) < 1e-2
