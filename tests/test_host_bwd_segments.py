"""Where the Mamba-2 backward splits a sequence of one forward segment (up to 16 chunks)
into finer segments, seen in its workspace query on the CPU: whole, it needs only the
log-decays, the totals and dg of its rows; split, also summaries and top-level states."""
import pytest

from hattention import _lib


@pytest.mark.parametrize("B,H", [(1, 1), (2, 4), (4, 8)])
@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 8, 11, 12, 16])
def test_short_sequences_stay_whole(chunks, B, H):
    T, rows = 64 * chunks, B * H
    need = _lib.load().hattn_mamba2_chunkwise_bwd_workspace(B, T, H, 64, 64, 11, 0)
    pad = lambda x: (x + 255) // 256 * 256
    whole = 2 * pad(rows * 4) + pad(B * T * H * 4)
    assert (need == whole) == (chunks < 12)
