"""Work that programs have this library do, as cases that can be timed and compared.

``listed()`` gives the fixed cases and ``draw(rng)`` one more of the same ranges; ``prepare`` makes what a program holds
before the call, ``run`` is one pass through the public ops, ``work`` what that pass cannot do without and
``tolerance`` how far another correct implementation at the same precision may be off.

Kinds of case:

``token``    one decode token of a Gated DeltaNet mixer between its projections: three short convolutions with their
             carry caches, the gate, the state step and the output norm -- six ops on a few kilobytes, the loop that a
             generating program runs per layer and token.
``step``     the state update of one decode token alone, fp32 state in place (delta / gated / kda / RWKV-7's dplr).
``forward``  a prompt: outputs and final state without gradients.  Up to 32 tokens go through the token-by-token op,
             longer prompts through the chunked one, the choice that the layers make.
``train``    forward and backward of a chunked op with gradients of every input, dense or packed sequences.
``scan``     forward and backward of the RWKV-7 scan (the layer trains through it).
``mixer``    forward and backward of the Gated DeltaNet or KDA mixer between its projections (convolutions, gate,
             chunked op on token-first views, output norm), the gradients of activations and parameters.
"""
from __future__ import annotations

import math

import torch

import linearnexus_amd as la

DEVICE = "cuda"
CHUNK = 64
CONV_TAPS = 4
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _case(kind, variant, B, H, T, dk, dv, dtype="bf16", *, nseq=0, l2norm=True, state=False, name=None):
    c = {"kind": kind, "variant": variant, "B": B, "H": H, "T": T, "dk": dk, "dv": dv, "dtype": dtype, "nseq": nseq,
         "l2norm": l2norm, "state": state}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one user's chat, one layer: latency and launches
        _case("token", "gated", 1, 16, 1, 128, 128, name="token_gated_b1"),
        # a server's ordinary batch, an odd number of sequences
        _case("step", "kda", 27, 16, 1, 128, 128, name="step_kda_b27"),
        # the repository's decode configuration: 512 MiB of state per token
        _case("step", "gated", 256, 32, 1, 128, 128, l2norm=False, name="step_gated_b256"),
        # one ordinary prompt, not a multiple of the chunk
        _case("forward", "gated", 1, 16, 1000, 128, 128, name="prompt_gated_t1000"),
        # one very long prompt, few heads
        _case("forward", "gated", 1, 4, 65536, 128, 128, l2norm=False, name="prompt_gated_t65536"),
        # a small model in the reference's default type at its own training batch, 8 x 128 tokens
        _case("mixer", "gated", 8, 4, 128, 64, 64, "f32", name="mixer_gated_f32_t128"),
        # a training micro-batch of ragged length through the whole mixer
        _case("mixer", "gated", 2, 16, 2007, 128, 128, name="mixer_gated_t2007"),
        # the repository's training configurations: gated (the headline), per-channel gate, packed sequences
        _case("train", "gated", 8, 16, 4096, 128, 128, l2norm=False, name="train_gated"),
        _case("train", "kda", 4, 16, 8192, 128, 128, state=True, name="train_kda"),
        _case("train", "delta", 1, 32, 32768, 128, 128, nseq=8, state=True, name="train_delta_packed"),
        # head shape of the Gated DeltaNet presets: keys of 256, values of 512
        _case("train", "gated", 8, 8, 4096, 256, 512, name="train_gated_dk256"),
        # RWKV-7 at its head size
        _case("scan", "dplr", 8, 16, 4096, 64, 64, name="scan_dplr"),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_MOST_TOKENS = 1 << 19  # head-tokens of a drawn case at dk = dv = 128, half of the largest listed case's


def draw(rng):
    kind = rng.choice(("token", "step", "step", "forward", "forward", "train", "train", "train", "scan", "mixer"))
    H = rng.choice((4, 6, 8, 12, 16, 32))
    dtype = "f32" if rng.random() < 0.25 else "bf16"
    if kind == "token":
        return _case(kind, "gated", _log_int(rng, 1, 64), H, 1, *rng.choice(((64, 64), (128, 128), (256, 512))), dtype)
    if kind == "step":
        variant = rng.choice(("delta", "gated", "kda", "dplr"))
        dk, dv = (64, 64) if variant == "dplr" else rng.choice(((64, 64), (128, 128), (256, 512)) if variant == "gated" else ((64, 64), (128, 128)))
        most = min(256, (1 << 27) // (H * dk * dv))
        return _case(kind, variant, _log_int(rng, 1, most), H, 1, dk, dv, dtype, l2norm=variant in ("gated", "kda"))
    if kind == "scan":
        T = _log_int(rng, 64, 4096)
        return _case(kind, "dplr", _log_int(rng, 1, min(16, max(1, (1 << 19) // (H * T)))), H, T, 64, 64, dtype, state=rng.random() < 0.3)
    if kind == "mixer":
        variant = rng.choice(("gated", "gated", "kda"))
    else:
        variant = rng.choice(("delta", "gated", "kda"))
    dk, dv = rng.choice(((64, 64), (128, 128), (128, 128), (256, 512)) if variant == "gated" else ((64, 64), (128, 128), (128, 128)))
    most = _MOST_TOKENS * 256 // (dk + dv) // (4 if dtype == "f32" else 1)
    T = _log_int(rng, 8 if kind == "forward" else 64, {"forward": 65536, "train": 16384, "mixer": 4096}[kind])
    B = _log_int(rng, 1, max(1, min(16, most // (H * T))))
    T = min(T, most // (B * H))
    nseq = 0
    if kind == "train" and T >= 512 and rng.random() < 0.3:
        T, B, nseq = B * T, 1, rng.randint(2, 12)
    return _case(kind, variant, B, H, T, dk, dv, dtype, nseq=nseq, l2norm=variant != "delta" and rng.random() < 0.7,
                 state=kind in ("forward", "train") and rng.random() < 0.4)


# ---- inputs ----

class _Rand:
    """Tensors of one seed, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device=DEVICE, dtype=torch.float32) * scale

    def unit(self, *shape):
        return torch.nn.functional.normalize(self.normal(*shape), dim=-1)

    def rate(self, *shape):  # learning rates
        return torch.sigmoid(self.normal(*shape))

    def decay(self, *shape, scale=0.1):  # log-decays <= 0
        return -torch.nn.functional.softplus(self.normal(*shape)) * scale


def _dplr_inputs(r, lead, dk, dv, dt):
    """What an RWKV-7 layer hands to the rule: the removal key and the in-context learning rate times it as a and b,
    decays between exp(-0.607) and 1."""
    kk = r.unit(*lead, dk)
    return {"q": r.normal(*lead, dk).to(dt), "k": r.normal(*lead, dk).to(dt), "v": r.normal(*lead, dv).to(dt),
            "a": (-kk).to(dt), "b": (kk * r.rate(*lead, dk)).to(dt), "gk": -0.606531 * r.rate(*lead, dk)}


def _lengths(seed, nseq, total):
    """cu_seqlens of nseq sequences that fill `total` tokens, of clearly different lengths."""
    gen = torch.Generator().manual_seed(seed)
    w = torch.rand(nseq, generator=gen) + 0.15
    edges = torch.cumsum(w / w.sum() * total, 0).round().to(torch.int32)
    edges[-1] = total
    return torch.cat([torch.zeros(1, dtype=torch.int32), edges]).to(DEVICE)


def _rule_inputs(r, c, lead, dt, seed):
    """q, k, v, beta, g, state of the delta rules for token tensors of the leading dimensions `lead`."""
    H, dk, dv = c["H"], c["dk"], c["dv"]
    # rows of length about sqrt(d) where the op normalises them, unit rows where the caller has done it
    rows = (lambda: r.normal(*lead, dk)) if c["l2norm"] else (lambda: r.unit(*lead, dk))
    x = {"q": rows().to(dt), "k": rows().to(dt), "v": r.normal(*lead, dv).to(dt), "beta": r.rate(*lead)}
    if c["variant"] == "gated":
        x["g"] = r.decay(*lead)
    elif c["variant"] == "kda":
        x["g"] = r.decay(*lead, dk, scale=0.05)
    if c["state"]:
        x["s0"] = r.normal(c["nseq"] or c["B"], H, dk, dv, scale=0.02)
    return x


def prepare(case, seed):
    c, r = case, _Rand(seed)
    dt = DTYPES[c["dtype"]]
    B, H, T, dk, dv, kind = c["B"], c["H"], c["T"], c["dk"], c["dv"], c["kind"]
    s = {"case": c}
    if kind == "token":
        act = lambda d: r.normal(B, 1, H * d).to(dt)
        s["x"] = {"q": act(dk), "k": act(dk), "v": act(dv), "gate": r.normal(B, H, dv).to(dt), "a": r.normal(B, 1, H), "b": r.normal(B, 1, H)}
        s["w"] = {"q": r.normal(CONV_TAPS, H * dk, scale=0.5), "k": r.normal(CONV_TAPS, H * dk, scale=0.5), "v": r.normal(CONV_TAPS, H * dv, scale=0.5),
                  "A_log": r.normal(H, scale=0.3), "dt_bias": r.normal(H, scale=0.3), "norm": 1.0 + r.normal(dv, scale=0.1)}
        s["cache"] = {n: r.normal(B, CONV_TAPS - 1, H * d).to(dt) for n, d in (("q", dk), ("k", dk), ("v", dv))}
        s["S"] = r.normal(B, H, dk, dv, scale=0.02)
        return s
    if kind == "step":
        s["x"] = _dplr_inputs(r, (B, H), dk, dv, dt) if c["variant"] == "dplr" else _rule_inputs(r, c, (B, H), dt, seed)
        s["S"] = r.normal(B, H, dk, dv, scale=0.02)
        return s
    if kind in ("forward", "train"):
        s["x"] = _rule_inputs(r, c, (B, H, T), dt, seed)
        s["cu"] = _lengths(seed, c["nseq"], T) if c["nseq"] else None
        # kda_chunkwise returns float32 whatever it is given, and the loss's gradient comes back in that type
        o_dt = torch.float32 if c["variant"] == "kda" else dt
    elif kind == "scan":
        s["x"] = _dplr_inputs(r, (B, H, T), dk, dv, dt)
        if c["state"]:
            s["x"]["s0"] = r.normal(B, H, dk, dv, scale=0.02)
        o_dt = dt
    else:
        gates = {"g_in": r.normal(B, T, H * dk).to(dt), "g_bias": r.normal(H * dk, scale=0.3)} if c["variant"] == "kda" \
            else {"a": r.normal(B, T, H), "dt_bias": r.normal(H, scale=0.3)}
        s["x"] = {"q": r.normal(B, T, H * dk).to(dt), "k": r.normal(B, T, H * dk).to(dt), "v": r.normal(B, T, H * dv).to(dt),
                  "gate": r.normal(B, T, H, dv).to(dt), "b": r.normal(B, T, H), "A_log": r.normal(H, scale=0.3) - 2.0,
                  "wq": r.normal(CONV_TAPS, H * dk, scale=0.5), "wk": r.normal(CONV_TAPS, H * dk, scale=0.5),
                  "wv": r.normal(CONV_TAPS, H * dv, scale=0.5), "norm": 1.0 + r.normal(dv, scale=0.1), **gates}
        o_dt = dt
    if kind != "forward":
        s["do"] = (r.normal(B, T, H, dv) if kind == "mixer" else r.normal(B, H, T, dv)).to(o_dt)
        for t in s["x"].values():
            t.requires_grad_(True)
    return s


# ---- passes ----

def _token(s):
    c, x, w, cache = s["case"], s["x"], s["w"], s["cache"]
    B, H, dk, dv = c["B"], c["H"], c["dk"], c["dv"]
    q, k, v = (la.depthwise_conv1d_causal(x[n], w[n], None, cache=cache[n], activation="silu", inplace_cache=True)[0] for n in ("q", "k", "v"))
    g, beta = la.gated_deltanet_gate(x["a"], w["A_log"], w["dt_bias"], x["b"])
    o, S = la.gated_delta_rule_step(q.view(B, H, dk), k.view(B, H, dk), v.view(B, H, dv), g.view(B, H), beta.view(B, H), s["S"], inplace=True)
    return la.rmsnorm_gated(o, x["gate"], w["norm"]), S, cache


def _step(s):
    c, x = s["case"], s["x"]
    if c["variant"] == "dplr":
        return la.dplr_delta_rule_step(x["q"], x["k"], x["v"], x["a"], x["b"], x["gk"], s["S"], inplace=True)
    if c["variant"] == "delta":
        return la.delta_rule_step(x["q"], x["k"], x["v"], x["beta"], s["S"], inplace=True)
    op = la.gated_delta_rule_step if c["variant"] == "gated" else la.kda_step
    return op(x["q"], x["k"], x["v"], x["g"], x["beta"], s["S"], None, c["l2norm"], inplace=True)


def _rule(s):
    c, x, cu = s["case"], s["x"], s["cu"]
    short = c["kind"] == "forward" and c["T"] <= 32
    q, k, v, beta, s0 = x["q"], x["k"], x["v"], x["beta"], x.get("s0")
    if c["variant"] == "delta":
        op = la.delta_rule_recurrent if short else la.delta_rule_chunkwise
        return op(q, k, v, beta, s0, cu_seqlens=cu)
    if short:
        op = la.gated_delta_rule_recurrent if c["variant"] == "gated" else la.kda_recurrent
        return op(q, k, v, x["g"], beta, None, s0, c["l2norm"])
    op = la.gated_delta_rule_chunkwise if c["variant"] == "gated" else la.kda_chunkwise
    return op(q, k, v, x["g"], beta, None, s0, CHUNK, c["l2norm"], cu_seqlens=cu)


def _mixer(s):
    c, x = s["case"], s["x"]
    B, H, T, dk, dv = c["B"], c["H"], c["T"], c["dk"], c["dv"]
    q, k, v = (la.depthwise_conv1d_causal(x[n], x["w" + n], None, activation="silu")[0] for n in ("q", "k", "v"))
    q, k, v = q.view(B, T, H, dk).transpose(1, 2), k.view(B, T, H, dk).transpose(1, 2), v.view(B, T, H, dv).transpose(1, 2)
    if c["variant"] == "kda":
        g, beta = la.kda_gate(x["g_in"], x["A_log"], dk, x["g_bias"], x["b"], out_dtype=torch.float32)
        o, S = la.kda_chunkwise(q, k, v, g.transpose(1, 2), beta.transpose(1, 2), output_dtype=q.dtype)
    else:
        g, beta = la.gated_deltanet_gate(x["a"], x["A_log"], x["dt_bias"], x["b"])
        o, S = la.gated_delta_rule_chunkwise(q, k, v, g.transpose(1, 2), beta.transpose(1, 2))
    return la.rmsnorm_gated(o.transpose(1, 2), x["gate"], x["norm"]), S


def run(state):
    s = state
    c, x = s["case"], s["x"]
    if c["kind"] == "token":
        return _token(s)
    if c["kind"] == "step":
        return _step(s)
    if c["kind"] == "forward":
        return _rule(s)
    if c["kind"] == "train":
        o, S = _rule(s)
    elif c["kind"] == "scan":
        o, S = la.dplr_delta_rule_recurrent(x["q"], x["k"], x["v"], x["a"], x["b"], x["gk"], c["dk"] ** -0.5, x.get("s0"))
    else:
        o, S = _mixer(s)
    grads = torch.autograd.grad(o, list(x.values()), s["do"])
    return o.detach(), S.detach(), grads


# ---- what a pass cannot do without ----

def work(case):
    c = case
    B, H, T, dk, dv, kind, variant = c["B"], c["H"], c["T"], c["dk"], c["dv"], c["kind"], c["variant"]
    n, es = B * H * T, DTYPES[c["dtype"]].itemsize
    nstate = (c["nseq"] or B) * H * dk * dv * 4
    gate = {"delta": 0, "gated": 1, "kda": dk, "dplr": dk}[variant] * 4
    if variant == "dplr":
        tok_in, rule = es * (4 * dk + dv) + gate, 9 * dk * dv * n
    else:
        tok_in = es * (2 * dk + dv) + 4 + gate
        # the chunk form's products per 64 tokens; a single token does 7 operations per state element
        rule = (2 * CHUNK * (3 * dk + 2 * dv) + 6 * dk * dv) * n if T > 32 else 7 * dk * dv * n
    o = (4 if variant == "kda" and kind in ("forward", "train", "step") else es) * dv
    if kind == "step":
        return {"bytes": n * (tok_in + o) + 2 * nstate, "flops": rule}
    width = H * (2 * dk + dv)  # channels of the three convolutions
    if kind == "token":
        conv = B * width * es * (2 * (CONV_TAPS - 1) + 1) + CONV_TAPS * width * 4
        return {"bytes": conv + n * (8 + es * dv + es * dv) + dv * 4 + 2 * nstate, "flops": rule + 2 * CONV_TAPS * B * width}
    if kind == "forward":
        return {"bytes": n * (tok_in + o) + nstate * (2 if c["state"] else 1), "flops": rule}
    if kind == "mixer":
        raw = es * dk if variant == "kda" else 4
        act = es * (2 * dk + 2 * dv) + raw + 4  # q, k, v, output gate; decay and learning-rate projections
        par = 4 * (CONV_TAPS * width + H + dv + (H * dk if variant == "kda" else H))
        return {"bytes": n * (2 * act + 2 * es * dv) + 2 * par + nstate, "flops": 3 * (rule + 2 * CONV_TAPS * B * T * width)}
    # train, scan: every input and the output gradient in; outputs, final state and the inputs' gradients out
    return {"bytes": n * (2 * tok_in + 2 * o) + nstate * (3 if c["state"] else 1), "flops": 3 * rule}


def tolerance(case):
    c = case
    if c["dtype"] == "f32" or (c["kind"] == "step" and c["variant"] == "kda"):  # kda_step: fp32 arithmetic, fp32 results
        return {"rel": 2e-5, "max": 2e-3}
    if c["kind"] in ("token", "step", "scan") or (c["kind"] == "forward" and c["T"] <= 32):
        return {"rel": 5e-3, "max": 5e-2}  # fp32 arithmetic between bf16 inputs and outputs
    return {"rel": 1e-2, "max": 0.3}  # bf16 operands of the matrix products
