"""An op gives the interpreter lock up while it allocates and launches, so that a call that waits for a full queue or for the driver
does not stop the program's other Python threads.  With a switch interval of minutes a waiting thread gets the lock only where
the running one gives it up by itself; the main thread does nothing but call the op."""
import sys
import threading
import time

import pytest
import torch

from linearnexus_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("name", ["step", "recurrent", "chunk", "chunk_segmented", "conv1d", "rmsnorm_gated", "gdn_gate", "kda_gate", "l2norm", "dplr", "dplr_step"])
def test_other_threads_run_during_an_op(name):
    host = _lib.host()
    r = lambda *s: torch.randn(*s, device=DEV)
    q, S, seq, gk = r(1, 2, 64) * 0.1, r(1, 2, 64, 64), r(1, 2, 64, 64) * 0.1, -r(1, 2, 64, 64).abs()
    beta, lead, x, w, ones = r(1, 2).sigmoid(), r(1, 2, 64).sigmoid(), r(1, 4, 64), r(4, 64), r(64)
    fn, args = {
        "step": (host.step, (q, q, q, None, beta, S, 0.125, False, False, True)),
        "recurrent": (host.recurrent, (seq, seq, seq, None, lead, None, 0.125, False, None)),
        "chunk": (host.chunk, (seq, seq, seq, None, lead, None, 0.125, False, 0, None, True, None, None, 0.0, 0, 0)),
        "chunk_segmented": (host.chunk_segmented, (seq, seq, seq, None, lead, None, 0.125, False, 0, 1)),
        "conv1d": (host.conv1d, (x, w, None, None, 0, False, None)),
        "rmsnorm_gated": (host.rmsnorm_gated, (seq, None, ones, 1e-5)),
        "gdn_gate": (host.gdn_gate, (lead, ones, None, None, 1.0)),
        "kda_gate": (host.kda_gate, (x, ones[:1], 64, None, None, 20.0, None)),
        "l2norm": (host.l2norm, (seq,)),
        "dplr": (host.dplr, (seq, seq, seq, seq, seq, gk, 0.1, None)),
        "dplr_step": (host.dplr_step, (q, q, q, q, q, gk[:, :, 0], S, 0.1, False)),
    }[name]
    fn(*args)
    torch.cuda.synchronize()
    ran, kept, go, old = [], [], threading.Event(), sys.getswitchinterval()

    def other():
        go.wait()
        ran.append(time.perf_counter())

    t = threading.Thread(target=other)
    t.start()
    time.sleep(0.05)  # the thread waits for the event
    try:
        sys.setswitchinterval(600)
        go.set()  # from here on the thread waits for the lock
        calls = 0
        while not ran and calls < 4_000:
            kept.append(fn(*args))  # a tensor's deallocation gives the lock up by itself
            calls += 1
        seen = bool(ran)
    finally:
        sys.setswitchinterval(old)
    t.join()
    torch.cuda.synchronize()
    print(f"the other thread ran after {calls} calls" if seen else f"not during {calls} calls")
    assert seen


@pytest.mark.parametrize("anomaly", [False, True])
def test_python_hooks_run_inside_the_ops(anomaly):
    """Saved-tensor hooks and the anomaly mode call into the interpreter while a node is made: they take the lock themselves."""
    import linearnexus_amd as la
    torch.manual_seed(0)
    r = lambda *s: torch.randn(*s, device=DEV).requires_grad_(True)
    B, T, H, d = 1, 70, 2, 64
    leaves = [r(B, T, H * d), r(4, H * d), r(B, T, H), r(H), r(B, T, H, d), r(d)]

    def loss():
        x, w, a, A_log, gate, norm = leaves
        y = la.depthwise_conv1d_causal(x, w, None, activation="silu")[0].view(B, T, H, d).transpose(1, 2)
        g, beta = la.gated_deltanet_gate(a, A_log, None, a)
        o, S = la.gated_delta_rule_chunkwise(y, y, y, g.transpose(1, 2), beta.transpose(1, 2))
        p, _ = la.dplr_delta_rule_recurrent(y, y, y, -y * 0.1, y * 0.1, -y.abs())
        return la.rmsnorm_gated((o + p).transpose(1, 2), gate, norm).square().sum() + S.square().sum()

    want = torch.autograd.grad(loss(), leaves)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.clone()

    with torch.autograd.set_detect_anomaly(anomaly), torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        got = torch.autograd.grad(loss(), leaves)
    assert len(packed) > 20
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4)
