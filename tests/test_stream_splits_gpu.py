"""The streaming kernels split their rows by the size of the call: the gate kernels by head count (heads that divide a
workgroup, that do not, more than one workgroup of them) and rows, the convolution's runs and the norm's steps by how many
waves there are, the parameter sums in one or two levels.  Every split against a plain torch restatement in fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(got, want, tol=1e-5):
    got, want = got.detach(), want.detach()
    e = float((got.double() - want.double()).abs().max() / want.double().abs().max().clamp_min(1e-30))
    assert e < tol, e


@pytest.mark.parametrize("rows,H", [(1, 1), (3, 5), (4014, 16), (300, 255), (65, 256), (9, 257), (5, 600), (70001, 6)])
def test_gdn_gate_rows_and_heads(rows, H):
    import linearnexus_amd as la
    torch.manual_seed(rows + H)
    r = lambda *s: torch.randn(*s, device=DEV)
    leaves = [r(rows, H), r(H) * 0.3, r(H) * 0.3, r(rows, H)]
    dg, db = r(rows, H), r(rows, H)
    x = [t.clone().requires_grad_(True) for t in leaves]
    y = [t.double().requires_grad_(True) for t in leaves]
    g, beta = la.gated_deltanet_gate(x[0], x[1], x[2], x[3])
    g64 = -torch.exp(y[1]) * torch.nn.functional.softplus(y[0] + y[2])
    b64 = torch.sigmoid(y[3])
    _close(g, g64), _close(beta, b64)
    got = torch.autograd.grad([g, beta], x, [dg, db])
    want = torch.autograd.grad([g64, b64], y, [dg.double(), db.double()])
    for a, b in zip(got, want):
        _close(a, b, 1e-4)


@pytest.mark.parametrize("rows,d", [(1, 64), (4096, 64), (33000, 128), (140001, 128), (9000, 384), (70000, 384)])
def test_rmsnorm_gated_steps_and_sums(rows, d):
    import linearnexus_amd as la
    torch.manual_seed(rows)
    r = lambda *s: torch.randn(*s, device=DEV)
    leaves, dy = [r(rows, d), r(rows, d), 1 + 0.1 * r(d)], r(rows, d)
    x = [t.clone().requires_grad_(True) for t in leaves]
    y = [t.double().requires_grad_(True) for t in leaves]
    o = la.rmsnorm_gated(*x)
    o64 = y[0] * torch.rsqrt((y[0] ** 2).mean(-1, keepdim=True) + 1e-5) * y[2] * torch.sigmoid(y[1])
    _close(o, o64)
    for a, b in zip(torch.autograd.grad(o, x, dy), torch.autograd.grad(o64, y, dy.double())):
        _close(a, b, 1e-4)


@pytest.mark.parametrize("B,T,D", [(1, 7, 16), (1, 65, 16), (8, 128, 256), (2, 501, 2048), (3, 2100, 1024), (8, 1030, 2048)])
def test_conv_runs(B, T, D):
    import linearnexus_amd as la
    torch.manual_seed(T)
    r = lambda *s: torch.randn(*s, device=DEV)
    leaves, dy = [r(B, T, D), r(4, D) * 0.5], r(B, T, D)
    x = [t.clone().requires_grad_(True) for t in leaves]
    y = [t.double().requires_grad_(True) for t in leaves]
    o, cache = la.depthwise_conv1d_causal(*x, activation="silu")
    p = torch.nn.functional.pad(y[0], (0, 0, 3, 0))
    o64 = torch.nn.functional.silu(sum(y[1][j] * p[:, j:j + T] for j in range(4)))
    _close(o, o64)
    assert torch.equal(cache, x[0].detach()[:, T - 3:])
    for a, b in zip(torch.autograd.grad(o, x, dy), torch.autograd.grad(o64, y, dy.double())):
        _close(a, b, 1e-4)
