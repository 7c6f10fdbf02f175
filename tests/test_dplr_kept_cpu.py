"""What the chunked RWKV-7 scan keeps between its passes: 48 KB per chunk of a (batch, head) row and one more state, no more."""
import pytest

from linearnexus_amd import _lib

LNX_DPLR_KEPT = 0


@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (1, 3, 64), (2, 2, 65), (8, 16, 4096)])
def test_kept_bytes(B, H, T):
    chunks = (T + 63) // 64
    assert _lib.load().lnx_dplr_chunk_bytes(B, H, T, LNX_DPLR_KEPT) == B * H * (48 * chunks + 16) * 1024
