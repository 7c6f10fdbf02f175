"""No op has a forward-mode derivative, and none may drop a tangent in silence: an input that carries one is refused, whether or not
a gradient is wanted, in grad mode and under no_grad."""
import pytest
import torch
from torch.autograd import forward_ad

import linearnexus_amd as la

DEV = "cuda"


def _calls():
    r = lambda *s: torch.randn(*s, device=DEV)
    B, H, T, d = 1, 2, 64, 64
    seq = dict(q=r(B, H, T, d), k=r(B, H, T, d), v=r(B, H, T, d), beta=r(B, H, T).sigmoid())
    long = dict(q=r(1, 4, 4160, d), k=r(1, 4, 4160, d), v=r(1, 4, 4160, d), beta=r(1, 4, 4160).sigmoid())
    tok = dict(q=r(B, H, d), k=r(B, H, d), v=r(B, H, d), beta=r(B, H).sigmoid(), state=r(B, H, d, d))
    dplr = dict(q=r(B, H, T, d), k=r(B, H, T, d), v=r(B, H, T, d), a=r(B, H, T, d), b=r(B, H, T, d), gk=-r(B, H, T, d).abs())
    dtok = dict(q=r(B, H, d), k=r(B, H, d), v=r(B, H, d), a=r(B, H, d), b=r(B, H, d), gk=-r(B, H, d).abs(), state=r(B, H, d, d))
    g, gv = dict(g=-r(B, H, T).abs()), dict(g=-r(B, H, T, d).abs())
    return {
        "conv": (lambda inputs, weight, bias, cache: la.depthwise_conv1d_causal(inputs, weight, bias, cache=cache, activation="silu"),
                 dict(inputs=r(B, T, 16), weight=r(4, 16), bias=r(16), cache=r(B, 3, 16))),
        "gated_deltanet_gate": (la.gated_deltanet_gate, dict(a=r(B, T, H), A_log=r(H), dt_bias=r(H), b=r(B, T, H))),
        "kda_gate": (lambda g, A_log, g_bias, beta: la.kda_gate(g, A_log, d, g_bias, beta), dict(g=r(B, T, H * d), A_log=r(H), g_bias=r(H * d), beta=r(B, T, H))),
        "rmsnorm_gated": (la.rmsnorm_gated, dict(x=r(B, T, H, d), gate=r(B, T, H, d), weight=r(d))),
        "l2norm_rows": (la.l2norm_rows, dict(x=r(B, H, T, d))),
        "delta_chunk": (la.delta_rule_chunkwise, seq),
        "gated_chunk": (la.gated_delta_rule_chunkwise, {**seq, **g}),
        "kda_chunk": (la.kda_chunkwise, {**seq, **gv}),
        "kda_chunk_raw_gate": (la.kda_chunkwise_raw_gate, dict(q=seq["q"], k=seq["k"], v=seq["v"], g_raw=r(B, H, T, d), beta=seq["beta"], A_log=r(H))),
        "delta_chunk_in_segments": (la.delta_rule_chunkwise, long),
        "delta_recurrent": (la.delta_rule_recurrent, seq),
        "gated_recurrent": (la.gated_delta_rule_recurrent, {**seq, **g}),
        "delta_step": (la.delta_rule_step, tok),
        "gated_step": (la.gated_delta_rule_step, {**tok, "g": -r(B, H).abs()}),
        "dplr_recurrent": (la.dplr_delta_rule_recurrent, dplr),
        "dplr_step": (la.dplr_delta_rule_step, dtok),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["plain", "requires_grad", "no_grad"])
@pytest.mark.parametrize("name", ["conv", "gated_deltanet_gate", "kda_gate", "rmsnorm_gated", "l2norm_rows", "delta_chunk", "gated_chunk", "kda_chunk",
                                  "kda_chunk_raw_gate", "delta_chunk_in_segments", "delta_recurrent", "gated_recurrent", "delta_step", "gated_step",
                                  "dplr_recurrent", "dplr_step"])
def test_tangents_are_refused(name, mode):
    op, x = _calls()[name]
    op(**x)  # the call itself is fine
    for carrier in x:
        with forward_ad.dual_level(), torch.set_grad_enabled(mode != "no_grad"):
            y = {n: (t.clone().requires_grad_(True) if mode == "requires_grad" else t) for n, t in x.items()}
            y[carrier] = forward_ad.make_dual(y[carrier], torch.ones_like(y[carrier]))
            with pytest.raises(RuntimeError, match="forward-mode|jvp"):
                op(**y)


@pytest.mark.gpu
def test_function_transforms_are_refused():
    x = torch.randn(2, 4, 64, device=DEV)
    with pytest.raises(RuntimeError):
        torch.func.jvp(la.l2norm_rows, (x,), (torch.ones_like(x),))
    with pytest.raises(RuntimeError):
        torch.func.vmap(la.l2norm_rows)(x)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["conv", "gated_deltanet_gate", "kda_gate", "rmsnorm_gated", "l2norm_rows", "gated_chunk", "dplr_recurrent"])
def test_tangents_of_output_gradients_are_refused(name):
    op, x = _calls()[name]
    x = {n: t.requires_grad_(True) for n, t in x.items()}
    y = op(**x)
    y = y if isinstance(y, torch.Tensor) else y[0]
    with forward_ad.dual_level():
        dy = forward_ad.make_dual(torch.ones_like(y), torch.ones_like(y))
        with pytest.raises(RuntimeError, match="forward-mode"):
            torch.autograd.grad(y, list(x.values()), dy, allow_unused=True)
