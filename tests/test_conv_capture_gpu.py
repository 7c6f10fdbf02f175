"""The convolution's parameter gradients in captured graphs: forward and backward each in a graph of its own (as
torch.cuda.make_graphed_callables records them), only one of the two captured, both in one graph.  The graphs are replayed in uneven
numbers with eager work in between, and every replay has to leave the eager gradients; gradients that an eager pass returned stay as
they are when the forward graph is replayed."""
import pytest
import torch

import linearnexus_amd as la

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs():
    torch.manual_seed(5)
    x, w, b = torch.randn(2, 150, 64, device=DEV), torch.randn(4, 64, device=DEV), torch.randn(64, device=DEV)
    return [t.requires_grad_(True) for t in (x, w, b)], torch.randn(2, 150, 64, device=DEV)


def _forward(leaves):
    return la.depthwise_conv1d_causal(leaves[0], leaves[1], leaves[2], activation="silu")[0]


def _backward(y, leaves, dy):
    return torch.autograd.grad(y, leaves, dy, retain_graph=True)


def _same(got, want):
    for g, e in zip(got, want):
        torch.testing.assert_close(g, e, rtol=1e-5, atol=1e-4)  # sums of 300 fp32 terms that are added in any order: 300 * 6e-8 * 5


def _capture(stream, fn):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = fn()
    return graph, out


@pytest.mark.parametrize("captured", ["both apart", "backward", "forward", "together"])
def test_every_replay_leaves_the_eager_gradients(captured):
    # a backward pass runs on the stream of its forward pass: all of the work below is on the one that captures
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        leaves, dy = _inputs()
        want = [g.clone() for g in _backward(_forward(leaves), leaves, dy)]
        torch.cuda.synchronize()
        if captured == "together":
            graph, got = _capture(stream, lambda: _backward(_forward(leaves), leaves, dy))
            for _ in range(3):
                graph.replay()
                _same(got, want)
                torch.cuda.synchronize()
            return
        if captured == "backward":
            y, replay = _forward(leaves), lambda: None
        else:
            fwd, y = _capture(stream, lambda: _forward(leaves))
            replay = fwd.replay
            replay()
        if captured == "forward":
            kept = _backward(y, leaves, dy)
            _same(kept, want)
            replay()
            _same(kept, want)  # the graph has not touched what the eager pass returned
            _same(_backward(y, leaves, dy), want)
            return
        torch.cuda.synchronize()
        bwd, got = _capture(stream, lambda: _backward(y, leaves, dy))
        for n in (1, 2, 3):
            replay()
            for _ in range(n):
                bwd.replay()
                _same(got, want)
                _same(_backward(_forward(leaves), leaves, dy), want)
            torch.cuda.synchronize()
