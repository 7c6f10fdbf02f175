"""dk = 256 through the direct-solve kernels (csrc/chunk_direct.hip, chunk_wide.hip): the L2 normalisation inside the kernels, value
dimensions whose slabs do not fill the ring of slab buffers evenly, and the rule that cuts a prompt into segments.  Bound 2e-2 of the largest
value against the fp64 oracles (bf16 inputs, fp32 accumulation)."""
import numpy as np
import pytest
import torch

from conftest import max_rel
from linearnexus_amd import _lib
from linearnexus_amd.linear_attn import _prefill_segments_256
from oracle.adjoint import delta_rule_adjoint
from oracle.inputs import make_inputs
from test_chunk_bwd_gpu import _prep, check, gpu_grads
from test_chunk_fwd_gpu import gpu_chunk_fwd, oracle_fwd


@pytest.mark.parametrize("H,T,dv,expected", [(4, 1984, 512, 1), (4, 1985, 512, 4), (4, 4032, 512, 4), (4, 4033, 512, 8), (5, 4096, 512, 8), (6, 4032, 512, 1),
                                             (6, 4096, 512, 4), (10, 8192, 512, 4), (11, 65536, 512, 1), (1, 16320, 512, 8), (2, 16384, 512, 16),
                                             (3, 32768, 512, 8)])
def test_segment_rule(monkeypatch, H, T, dv, expected):
    monkeypatch.delenv("LNX_PREFILL_SEGMENTS", raising=False)
    assert _prefill_segments_256(1, H, T, dv) == expected
    monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "3")
    assert _prefill_segments_256(1, H, T, dv) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("dv", [64, 128, 320])  # two, four and ten slabs through three buffers
@pytest.mark.parametrize("T,packed", [(1, False), (130, False), (200, True)])
def test_l2norm_inside(dv, T, packed):
    B, H, dk = (1 if packed else 2), 2, 256
    x = make_inputs(91, B, H, T, dk, dv, gate="scalar", with_state=not packed, with_grad=True, normalize=False)
    rng = np.random.default_rng(92)
    for n in "qk":
        x[n] = x[n] * np.exp(rng.standard_normal((B, H, T, 1))).astype(np.float32)
    a = _lib.ScanArgs(B=B, H=H, T=T, dk=dk, dv=dv, chunk=64, dtype=_lib.LNX_BF16, o_dtype=_lib.LNX_BF16, gate=_lib.GATE_SCALAR)
    assert _lib.load().lnx_chunk_fuses_l2norm(a) == 1
    cu = np.array([0, 3, 70, T], np.int32) if packed else None
    if packed:
        x["S0"], x["dS"] = ((rng.standard_normal((3, H, dk, dv)) * s).astype(np.float32) for s in (0.02, 0.1))
    x, dt = _prep(x, True)
    if not packed:
        o_ref, S_ref = oracle_fwd(x, "scalar", l2=True)
        with torch.no_grad():
            o, S = gpu_chunk_fwd(x, "scalar", dt, l2=True)
        assert max_rel(o.float().cpu().numpy(), o_ref) < 2e-2 and max_rel(S.cpu().numpy(), S_ref) < 2e-2
    spans = list(zip(cu[:-1], cu[1:])) if packed else [(0, T)]
    parts = [delta_rule_adjoint(*(x[n][:, :, lo:hi] for n in ("q", "k", "v", "beta", "dO", "g")), x["dS"][i:i + 1] if packed else x["dS"], None,
                                x["S0"][i:i + 1] if packed else x["S0"], True) for i, (lo, hi) in enumerate(spans)]
    ref = {n: np.concatenate([p[n] for p in parts], 2) for n in ("dq", "dk", "dv", "dbeta", "dg")}
    ref["dS0"] = np.concatenate([p["dS0"] for p in parts], 0)
    check(gpu_grads(x, "scalar", dt, cu=cu, l2=True), ref, 2e-2)
