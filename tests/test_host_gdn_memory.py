"""What a Gated DeltaNet training call with V outside {64, 128} holds and takes, by the
host's rules, on the CPU."""
import pytest

from hattention import _lib, chunkwise_hgdn as hg


@pytest.mark.parametrize("shape,cols,keeps", [
    ((1, 16384, 6, 192, 384, 15), 384, True),
    ((8, 8192, 16, 256, 512, 14), 128, False),
    ((2, 8192, 8, 256, 512, 14), 256, False),
    ((1, 64, 1, 64, 192, 7), 192, True),
    ((8, 8192, 16, 256, 128, 14), 128, False)])
def test_columns_and_kept_workspace(shape, cols, keeps):
    lib = _lib.load()
    B, T, H, K, V, L = shape
    assert hg.bwd_columns(*shape) == cols
    assert hg.keeps_workspace(*shape) == keeps
    need = lambda n: lib.hattn_gdn_chunkwise_bwd_workspace(B, T, H, K, n, L)
    if cols > hg.VB:
        assert need(cols) <= hg.BWD_LIMIT
    if cols < V:
        assert need(cols + hg.VB) > hg.BWD_LIMIT
