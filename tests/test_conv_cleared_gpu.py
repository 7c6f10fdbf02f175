"""The convolution's parameter gradients add to a buffer that the forward kernel cleared: the first backward pass of a node takes
it, later ones (retain_graph) bring their own, all with the same gradients; sizes down to one token, empty inputs, packed batches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,D,K,bias,packed", [(1, 1, 8, 4, True, False), (2, 37, 264, 4, False, False), (1, 70, 64, 3, True, True), (2, 0, 16, 4, True, False), (3, 9, 8, 1, True, False)])
def test_gradients_of_repeated_backward_passes(B, T, D, K, bias, packed):
    import linearnexus_amd as la
    torch.manual_seed(D)
    x = torch.randn(B, T, D, device="cuda", requires_grad=True)
    w = torch.randn(K, D, device="cuda", requires_grad=True)
    b = torch.randn(D, device="cuda", requires_grad=True) if bias else None
    cu = torch.tensor([0, 30, 31, T], dtype=torch.int32, device="cuda") if packed else None
    y = la.depthwise_conv1d_causal(x, w, b, activation="silu", **({"cu_seqlens": cu} if packed else {}))[0]
    dy = torch.randn_like(y)
    leaves = [t for t in (x, w, b) if t is not None]
    first = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    kept = [g.clone() for g in first]
    again = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    torch.autograd.grad(y, leaves, 2 * dy)
    for f, k, a in zip(first, kept, again):
        assert torch.equal(f, k)  # nobody writes into the first pass's gradients
        torch.testing.assert_close(a, k, rtol=1e-5, atol=1e-5)
    if T:
        if not packed and K > 1:
            xd, wd = x.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
            z = torch.nn.functional.conv1d(torch.nn.functional.pad(xd.transpose(1, 2), (K - 1, 0)), wd.t().unsqueeze(1), None if b is None else b.detach().double(), groups=D)
            gx, gw = torch.autograd.grad(torch.nn.functional.silu(z).transpose(1, 2), [xd, wd], dy.double())
            torch.testing.assert_close(kept[0].double(), gx, rtol=1e-4, atol=1e-4)
            torch.testing.assert_close(kept[1].double(), gw, rtol=1e-4, atol=1e-4)
    else:
        assert not kept[1].any()
