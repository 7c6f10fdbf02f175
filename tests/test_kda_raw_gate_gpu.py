"""kda_chunkwise_raw_gate: the KDA block's gate activation (kda_gate, kda.py:120-172) inside the chunk op (kda.py:350-655).
Oracle: oracle.gate.kda_gate composed with the fp64 token-by-token KDA scan, and for the gradients the scan's
token-level adjoint followed by oracle.gate.kda_gate_grad.  Tolerances max|x - ref| / max|ref|: 1e-4 for fp32 inputs,
2e-2 for bf16 inputs (fp32 accumulation)."""
import numpy as np
import pytest
import torch

from oracle import gate as og
from oracle import recurrent as rc
from oracle.adjoint import delta_rule_adjoint
from oracle.inputs import make_inputs, to_bf16_grid
from conftest import max_rel

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(seed, B, H, T, dk, dv, bf16, bias, cu=None):
    x = make_inputs(seed, B, H, T, dk, dv, gate="vector", with_state=cu is None, with_grad=True)
    r = np.random.default_rng(seed + 1)
    rnd = (lambda a: to_bf16_grid(a.astype(np.float32))) if bf16 else (lambda a: a.astype(np.float32))
    for n in ("q", "k", "v", "dO"):
        x[n] = rnd(x[n])
    # raw projection [B, T, H * dk]; x = raw + bias around -3 .. 1 keeps the decays per token between about 0.3 and 1
    x["raw"] = rnd(r.standard_normal((B, T, H * dk)) - 2.0)
    x["A_log"] = (r.standard_normal(H) * 0.3 - 1.0).astype(np.float32)
    x["bias"] = (r.standard_normal(H * dk) * 0.5).astype(np.float32) if bias else None
    return x


def _oracle(x, dk, thr, S0=None, dS=None):
    g4, _ = og.kda_gate(x["raw"], x["A_log"], dk, x["bias"], None, thr)          # [B,T,H,dk]
    g = np.ascontiguousarray(g4.transpose(0, 2, 1, 3))
    o, S = rc.kda_recurrent(x["q"], x["k"], x["v"], g, x["beta"], None, S0, False)
    ref = delta_rule_adjoint(x["q"], x["k"], x["v"], x["beta"], x["dO"], g, dS, None, S0, False)
    draw, dA, dbias = og.kda_gate_grad(x["raw"], x["A_log"], dk, ref["dg"].transpose(0, 2, 1, 3), x["bias"], thr)
    return o, S, ref, draw, dA, dbias


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("shape", [(2, 2, 150, 128, 128), (1, 3, 64, 64, 64), (1, 2, 200, 256, 128)])
def test_raw_gate_forward_backward_match_oracle(shape, bias, bf16):
    import linearnexus_amd as la
    B, H, T, dk, dv = shape
    thr = 0.5  # some entries of raw + bias lie above it: the linear branch of softplus is exercised
    x = _case(101, B, H, T, dk, dv, bf16, bias)
    o_ref, S_ref, ref, draw_ref, dA_ref, dbias_ref = _oracle(x, dk, thr, x["S0"], x["dS"])
    dt = torch.bfloat16 if bf16 else torch.float32
    t = lambda a, d=None, g=True: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(d or torch.float32).requires_grad_(g)
    q, k, v = t(x["q"], dt), t(x["k"], dt), t(x["v"], dt)
    raw = t(x["raw"], dt)                                       # [B, T, H*dk], the projection's layout
    beta, S0, A = t(x["beta"]), t(x["S0"]), t(x["A_log"])
    gb = t(x["bias"]) if bias else None
    g_view = raw.view(B, T, H, dk).transpose(1, 2)              # [B, H, T, dk] on token-first memory
    # q, k, v head-first and the gate token-first is not one layout: bring the gate to q's layout like a caller would
    o, S = la.kda_chunkwise_raw_gate(q, k, v, g_view.contiguous(), beta, A, gb, None, S0, 64, False, threshold=thr)
    assert o.dtype == torch.float32  # kda.py:655
    tol = 2e-2 if bf16 else 1e-4
    assert max_rel(o.detach().cpu().numpy(), o_ref) < tol and max_rel(S.detach().cpu().numpy(), S_ref) < tol
    ((o * t(x["dO"], None, False)).sum() + (S * t(x["dS"], None, False)).sum()).backward()
    f = lambda z: z.grad.float().cpu().numpy()
    for name, leaf in (("dq", q), ("dk", k), ("dv", v), ("dbeta", beta), ("dS0", S0)):
        assert max_rel(f(leaf), ref[name]) < tol, name
    assert max_rel(f(raw), draw_ref) < tol
    assert max_rel(f(A), dA_ref) < tol
    if bias:
        assert max_rel(f(gb), dbias_ref) < tol


def test_raw_gate_token_first_views_and_packed_batch_and_determinism():
    """[B,T,H,.] projections used in place through transposed views; a packed batch with an unused chunk slot per
    sequence boundary; two backward passes give bit-identical parameter gradients (no atomics)."""
    import linearnexus_amd as la
    H, T, d, thr = 3, 300, 128, 20.0
    cu = [0, 70, 70, 199, 300]
    x = _case(102, 1, H, T, d, d, True, True, cu=cu)
    t = lambda a, dt=None, g=True: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(dt or torch.float32).requires_grad_(g)
    tf = lambda a: t(a.transpose(0, 2, 1, 3), torch.bfloat16)   # [1, T, H, d] leaves
    q, k, v = tf(x["q"]), tf(x["k"]), tf(x["v"])
    raw = t(x["raw"], torch.bfloat16)
    beta, A, gb = t(x["beta"].transpose(0, 2, 1)), t(x["A_log"]), t(x["bias"])
    dO = t(x["dO"], None, False)
    grads = []
    for _ in range(2):
        for z in (q, k, v, raw, beta, A, gb):
            z.grad = None
        o, S = la.kda_chunkwise_raw_gate(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2),
                                         raw.view(1, T, H, d).transpose(1, 2), beta.transpose(1, 2), A, gb, None, None, 64,
                                         False, threshold=thr, cu_seqlens=cu)
        (o * dO).sum().backward()
        grads.append([z.grad.clone() for z in (q, k, v, raw, beta, A, gb)])
    for a, b in zip(*grads):
        assert torch.equal(a, b)
    # oracle: one scan per sequence
    g4, _ = og.kda_gate(x["raw"], x["A_log"], d, x["bias"], None, thr)
    g = np.ascontiguousarray(g4.transpose(0, 2, 1, 3))
    o_ref = np.zeros_like(x["v"], dtype=np.float64)
    dg = np.zeros_like(g)
    refs = {n: np.zeros_like(x[s], dtype=np.float64) for n, s in (("dq", "q"), ("dk", "k"), ("dv", "v"), ("dbeta", "beta"))}
    for a, b in zip(cu[:-1], cu[1:]):
        if a == b:
            continue
        sl = lambda z: z[:, :, a:b]
        o_ref[:, :, a:b], _ = rc.kda_recurrent(sl(x["q"]), sl(x["k"]), sl(x["v"]), sl(g), sl(x["beta"]), None, None, False)
        r = delta_rule_adjoint(sl(x["q"]), sl(x["k"]), sl(x["v"]), sl(x["beta"]), sl(x["dO"]), sl(g), None, None, None, False)
        dg[:, :, a:b] = r["dg"]
        for n in refs:
            refs[n][:, :, a:b] = r[n]
    draw_ref, dA_ref, dbias_ref = og.kda_gate_grad(x["raw"], x["A_log"], d, dg.transpose(0, 2, 1, 3), x["bias"], thr)
    assert max_rel(o.detach().cpu().numpy(), o_ref) < 2e-2
    gq, gk, gv, graw, gbeta, gA, gbias = grads[0]
    hf = lambda z: z.float().cpu().numpy().transpose(0, 2, 1, 3)
    assert max_rel(hf(gq), refs["dq"]) < 2e-2 and max_rel(hf(gk), refs["dk"]) < 2e-2 and max_rel(hf(gv), refs["dv"]) < 2e-2
    assert max_rel(gbeta.cpu().numpy().transpose(0, 2, 1), refs["dbeta"]) < 2e-2
    assert max_rel(graw.float().cpu().numpy(), draw_ref) < 2e-2
    assert max_rel(gA.cpu().numpy(), dA_ref) < 2e-2 and max_rel(gbias.cpu().numpy(), dbias_ref) < 2e-2


def test_raw_gate_equals_gate_kernel_then_scan_and_refuses_bad_arguments():
    import linearnexus_amd as la
    B, H, T, d = 2, 2, 130, 128
    x = _case(103, B, H, T, d, d, True, True)
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(dt or torch.float32)
    q, k, v, raw = (t(x[n], torch.bfloat16) for n in ("q", "k", "v", "raw"))
    beta, A, gb = t(x["beta"]), t(x["A_log"]), t(x["bias"])
    gv = raw.view(B, T, H, d).transpose(1, 2).contiguous()
    o1, S1 = la.kda_chunkwise_raw_gate(q, k, v, gv, beta, A, gb)             # use_qk_l2norm=True, the reference's default
    g, _ = la.kda_gate(raw, A, d, gb, out_dtype=torch.float32)
    o2, S2 = la.kda_chunkwise(q, k, v, g.transpose(1, 2), beta)
    assert (o1 - o2).abs().max() <= 1e-5 * o2.abs().max() and (S1 - S2).abs().max() <= 1e-5 * S2.abs().max()
    with pytest.raises(ValueError):
        la.kda_chunkwise_raw_gate(q, k, v, gv, beta, A, gb, chunk_size=24)
    with pytest.raises(RuntimeError):
        la.kda_chunkwise_raw_gate(q, k, v, gv.float(), beta, A, gb)          # gate dtype differs from q's
    with pytest.raises(RuntimeError):
        la.kda_chunkwise_raw_gate(q, k, v, gv, beta, A[:1], gb)


@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("B,H,T,dv,cu", [(2, 3, 256, 64, None), (2, 3, 253, 128, None), (8, 8, 637, 64, None), (1, 3, 317, 64, [0, 61, 61, 189, 317])])
def test_raw_gate_gradients_dk64(B, H, T, dv, cu, bias, l2):
    """bf16 with dk = 64, where the gate's gradient on its way out and its partial sums share the place of the tiles: full chunks, 61 and 62 tokens
    left, more chunks than fit the GPU at once, a packed batch with an empty sequence; the chunks' last four tokens by themselves, and the
    same bits twice."""
    import linearnexus_amd as la
    dk, thr = 64, 0.5
    x = _case(104, B, H, T, dk, dv, True, bias, cu=cu)
    if l2:
        for n in "qk":
            x[n] = to_bf16_grid(x[n] * np.exp(np.random.default_rng(105).standard_normal((B, H, T, 1))).astype(np.float32))
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(dt or torch.float32).requires_grad_()
    q, k, v = (t(x[n], torch.bfloat16) for n in "qkv")
    raw = t(x["raw"].reshape(B, T, H, dk).transpose(0, 2, 1, 3), torch.bfloat16)
    leaves = [q, k, v, raw, t(x["beta"]), t(x["A_log"])] + ([t(x["bias"])] if bias else [])
    q, k, v, raw, beta, A = leaves[:6]
    dO = torch.from_numpy(x["dO"]).to(DEV)
    runs = []
    for _ in range(2):
        o, _ = la.kda_chunkwise_raw_gate(q, k, v, raw, beta, A, leaves[6] if bias else None, None, None, 64, l2, threshold=thr, cu_seqlens=cu)
        runs.append(torch.autograd.grad((o * dO).sum(), leaves))
    for a, b in zip(*runs):
        assert torch.equal(a, b)
    g = np.ascontiguousarray(og.kda_gate(x["raw"], x["A_log"], dk, x["bias"], None, thr)[0].transpose(0, 2, 1, 3))
    spans = [(a, b) for a, b in zip(cu[:-1], cu[1:]) if a < b] if cu else [(0, T)]
    parts = [delta_rule_adjoint(*(z[:, :, a:b] for z in (x["q"], x["k"], x["v"], x["beta"], x["dO"], g)), None, None, None, l2) for a, b in spans]
    ref = {n: np.concatenate([r[n] for r in parts], 2) for n in ("dq", "dk", "dv", "dg", "dbeta")}
    draw = og.kda_gate_grad(x["raw"], x["A_log"], dk, ref["dg"].transpose(0, 2, 1, 3), x["bias"], thr)[0].reshape(B, T, H, dk).transpose(0, 2, 1, 3)
    got = [z.double().cpu().numpy() for z in runs[0]]
    for a, b in zip(got, (ref["dq"], ref["dk"], ref["dv"], draw, ref["dbeta"])):
        assert max_rel(a, b) < 2e-2
    last = np.concatenate([np.arange(c + min(60, b - c), min(c + 64, b)) for a, b in spans for c in range(a, b, 64)])
    assert max_rel(got[3][:, :, last], draw[:, :, last]) < 2e-2
    # The parameters' gradients are sums of thousands of terms of either sign, so they are held to the op's own d_raw: its values are the summed
    # ones rounded to bf16, an error of 2^-9 / sqrt(3) of a term at most in the mean (eight standard deviations), beside the fp32 sums.
    z = x["raw"].astype(np.float64).reshape(B, T, H, dk).transpose(0, 2, 1, 3) + (x["bias"].reshape(H, 1, dk) if bias else 0.0)
    lin = z > thr
    to_A = np.where(lin, z, np.log1p(np.exp(np.minimum(z, thr)))) * np.where(lin, 1.0, 1.0 + np.exp(-z))  # softplus over its derivative
    sums = [(got[5], got[3] * to_A, (0, 2, 3))] + ([(got[6].reshape(H, dk), got[3], (0, 2))] if bias else [])
    for total, terms, axes in sums:
        bound = 8 * 2.0 ** -9 / 3 ** 0.5 * np.sqrt((terms ** 2).sum(axes)) + 1e-5 * np.abs(terms).sum(axes)
        assert (np.abs(total - terms.sum(axes)) <= bound).all()
