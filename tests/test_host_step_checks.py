"""Operands whose length does not fit are refused before any launch (the kernels index them
by head and token): checked on the CPU, where everything after the checks is refused too,
as no HIP device."""
import pytest
import torch

from hattention.base import HStruct, HType
from hattention.recurrent import HState


@pytest.mark.parametrize("n", [1, 3, 5])
@pytest.mark.parametrize("which", ["A", "dt_bias", "D"])
def test_layer_step_per_head_operands(which, n):
    from hattention.mamba_apis import hselective_state_update
    B, H, P, N, L = 2, 4, 64, 64, 9
    S = HState(2, HType.WEAK, HStruct.MAMBA2, (B, H, N, P, L), torch.float32, "cpu")
    par = {w: torch.zeros(H) for w in ("A", "dt_bias", "D")}
    par[which] = torch.zeros(n)
    with pytest.raises(ValueError):
        hselective_state_update(
            S, torch.zeros(B, H, P), torch.zeros(B, H), par["A"], torch.zeros(B, 1, N),
            torch.zeros(B, 1, N), torch.zeros(B, H, L), torch.zeros(H, L), D=par["D"],
            dt_bias=par["dt_bias"], dt_softplus=True, lambda_mode="positive", lambda_level_max=L,
            lambda_level_base=2, lambda_htype=HType.WEAK, lambda_hstruct=HStruct.MAMBA2,
            lambda_level_fixed=True)


@pytest.mark.parametrize("shape", [(1, 64, 2), (2, 63, 2), (2, 64, 1), (2, 64), (256,)])
def test_prefill_levels_beta(shape):
    from hattention.kernel import postprocess_prefill_hstate_
    B, T, H, K, V, L = 2, 64, 2, 64, 64, 9
    S = HState(2, HType.WEAK, HStruct.GDELTA, (B, H, K, V, L), torch.float32, "cpu")
    z = torch.zeros
    with pytest.raises(ValueError):
        postprocess_prefill_hstate_(
            hstate=S, q=z(B, T, H, K), k=z(B, T, H, K), v=z(B, T, H, V), b=z(*shape), g=z(B, T, H),
            l=z(B, T, H, L), scale=1.0, head_first=False, level_base=2, htype=HType.WEAK,
            hstruct=HStruct.GDELTA, chunk_size=64, use_qk_l2norm_in_kernel=True)
