"""The final state of a prompt that is cut into segments holds its own memory and not that of every segment's state: a program that
caches it keeps what one chain's call would have it keep."""
import pytest
import torch

import linearnexus_amd as la

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,H", [(1, 4), (2, 2)])
@pytest.mark.parametrize("variant", ["delta", "gated", "kda"])
def test_final_state_owns_its_memory(variant, B, H, monkeypatch):
    torch.manual_seed(2)
    T, d = 8257, 128
    q, k = (torch.nn.functional.normalize(torch.randn(B, H, T, d, device=DEV), dim=-1).bfloat16() for _ in "qk")
    v, beta = torch.randn(B, H, T, d, device=DEV).bfloat16(), torch.rand(B, H, T, device=DEV)
    g = -0.01 * torch.rand(*((B, H, T, d) if variant == "kda" else (B, H, T)), device=DEV)
    op = {"delta": la.delta_rule_chunkwise, "gated": la.gated_delta_rule_chunkwise, "kda": la.kda_chunkwise}[variant]

    def run():
        with torch.no_grad():
            return op(q, k, v, *(() if variant == "delta" else (g,)), beta)

    o, S = run()
    held = S.untyped_storage().nbytes()  # a number: an assertion would print the storage byte by byte
    assert S.shape == (B, H, d, d) and S.is_contiguous() and held == S.numel() * 4
    monkeypatch.setenv("LNX_PREFILL_SEGMENTS", "1")
    o1, S1 = run()
    assert (S - S1).norm() < 2e-2 * S1.norm() and (o.float() - o1.float()).norm() < 2e-2 * o1.float().norm()


@pytest.mark.parametrize("dtype,dk", [(torch.bfloat16, 128), (torch.bfloat16, 256), (torch.float32, 64)])
def test_states_of_all_segments_through_the_c_abi(dtype, dk):
    """lnx_chunk_fwd_segmented gives the state at every segment's end; the last one, bit for bit, is what the other entry point gives."""
    import ctypes as C

    from linearnexus_amd import _lib
    lib = _lib.load()
    lib.lnx_chunk_fwd_segmented_bytes.restype = C.c_uint64
    torch.manual_seed(4)
    H, T, dv, n = 3, 1000, 128, 4
    q, k = (torch.nn.functional.normalize(torch.randn(1, H, T, dk, device=DEV), dim=-1).to(dtype) for _ in "qk")
    v, beta, s0 = torch.randn(1, H, T, dv, device=DEV).to(dtype), torch.rand(1, H, T, device=DEV), torch.randn(1, H, dk, dv, device=DEV)
    code = 1 if dtype == torch.bfloat16 else 0
    a = _lib.ScanArgs(B=1, H=H, T=T, dk=dk, dv=dv, chunk=64, dtype=code, o_dtype=code, gate=0, scale=0.1, forward_only=1)
    for name, t in (("q", q), ("k", k), ("v", v), ("beta", beta), ("initial_state", s0)):
        setattr(a, name, t.data_ptr())
    ws = torch.empty(int(lib.lnx_chunk_fwd_segmented_bytes(C.byref(a), n)), dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    outs = {}
    for fn, states in (("lnx_chunk_fwd_segmented", n), ("lnx_chunk_fwd_segmented_final", 1)):
        o, S = torch.full((1, H, T, dv), float("nan"), device=DEV, dtype=dtype), torch.full((states + 1, H, dk, dv), float("nan"), device=DEV)
        a.o, a.final_state = o.data_ptr(), S.data_ptr()
        assert getattr(lib, fn)(C.byref(a), C.c_int32(n), stream) == 0
        torch.cuda.synchronize()
        assert torch.isfinite(S[:states]).all() and torch.isnan(S[states]).all()  # and not a byte more
        outs[states] = o, S[states - 1]
    assert torch.equal(outs[n][0], outs[1][0]) and torch.equal(outs[n][1], outs[1][1])
    import linearnexus_amd as la
    with torch.no_grad():
        o, S = la.delta_rule_chunkwise(q, k, v, beta, s0, 64, 0.1)
    assert (outs[1][0].float() - o.float()).norm() < 2e-2 * o.float().norm() and (outs[1][1] - S[0]).norm() < 2e-2 * S.norm()
