"""hselective_state_update (one hattn_mamba2_layer_step launch) against the same step
from its parts, layer_prologue -> launch_step -> layer_epilogue: the same bits, for
every dtype mix, lambda mode and optional operand, and at the sizes where the state
kernel takes another lane width or leaves a block part empty."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32


def _run(B, H, P, N, G, L, act, par, mode, bias, resid, strong=False):
    from hattention.base import HStruct, HType
    from hattention.mamba_apis import hselective_state_update
    from hattention.mamba_layer import layer_epilogue, layer_prologue
    from hattention.recurrent import HState, launch_step
    print(f"[layer step] B={B} H={H} P={P} N={N} G={G} L={L} {act} {par} {mode} {bias} {resid}", flush=True)
    htype = HType.STRONG if strong else HType.WEAK
    gen = torch.Generator(DEV).manual_seed(B * 100 + L)
    rn = lambda *s, dtype=act: torch.randn(*s, device=DEV, generator=gen).to(dtype)
    S, R = (HState(2, htype, HStruct.MAMBA2, (B, H, N, P, L), F32, DEV) for _ in range(2))
    A, Lp = -torch.rand(H, device=DEV, generator=gen), rn(H, L, dtype=par)
    D, db = rn(H, dtype=par) if resid else None, rn(H, dtype=par) if bias else None
    for _ in range(min(6, 2 ** (L - 1))):
        x, dt, dl = rn(B, H, P), rn(B, H), rn(B, H, L)
        Bm, Cm = rn(B, G, N), rn(B, G, N)
        out, S = hselective_state_update(
            S, x, dt, A, Bm, Cm, dl, Lp, D=D, dt_bias=db, dt_softplus=True, lambda_mode=mode,
            lambda_level_max=L, lambda_level_base=2, lambda_htype=htype,
            lambda_hstruct=HStruct.MAMBA2, lambda_level_fixed=True)
        v, g, lam = layer_prologue(x.unsqueeze(1), dt.unsqueeze(1), A, db, dl.unsqueeze(1), Lp, True, mode)
        ref = torch.empty_like(v.squeeze(1))
        launch_step(R, q=Cm, k=Bm, v=v.squeeze(1), g=g.squeeze(1), l=lam.squeeze(1), o=ref,
                    update=True, output=True)
        if resid:
            ref = layer_epilogue(ref.unsqueeze(1), x.unsqueeze(1), D).squeeze(1)
        assert out.dtype == ref.dtype and torch.equal(out, ref)
        assert torch.equal(S.states, R.states) and torch.equal(S.counts, R.counts)
        assert S.host_counts == R.host_counts


@pytest.mark.parametrize("bias,resid", [(False, False), (True, True)])
@pytest.mark.parametrize("mode", ["positive", "bounded", None])
@pytest.mark.parametrize("act,par", [(BF, BF), (BF, F32), (F32, F32)])
def test_layer_step_types(act, par, mode, bias, resid):
    _run(2, 4, 64, 64, 2, 9, act, par, mode, bias, resid)


@pytest.mark.parametrize("B,H,P,N,G,L", [(1, 1, 16, 16, 1, 1), (1, 3, 32, 100, 3, 7), (64, 16, 64, 64, 1, 18),
                                         (48, 16, 128, 128, 4, 19), (2, 2, 256, 256, 2, 32)])
def test_layer_step_sizes(B, H, P, N, G, L):
    _run(B, H, P, N, G, L, BF, BF, "positive", True, True)
    _run(B, H, P, N, G, L, BF, BF, "positive", True, True, strong=True)


@pytest.mark.parametrize("which", ["A", "dt_bias", "D"])
def test_layer_step_half_parameters(which):
    """fp16 per-head parameters are taken as their fp32 values."""
    from hattention.base import HStruct, HType
    from hattention.mamba_apis import hselective_state_update
    from hattention.recurrent import HState
    print(f"[layer step] fp16 {which}", flush=True)
    B, H, P, N, L = 2, 4, 64, 64, 9
    gen = torch.Generator(DEV).manual_seed(3)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    x, dt, dl, Lp = rn(B, H, P), rn(B, H), rn(B, H, L), rn(H, L)
    Bm, Cm = rn(B, 1, N), rn(B, 1, N)
    par = dict(A=-rn(H).abs(), dt_bias=rn(H), D=rn(H))
    half = dict(par, **{which: par[which].half()})
    outs = []
    for p in (half, {n: t.float() for n, t in half.items()}):
        S = HState(2, HType.WEAK, HStruct.MAMBA2, (B, H, N, P, L), F32, DEV)
        out, S = hselective_state_update(
            S, x, dt, p["A"], Bm, Cm, dl, Lp, D=p["D"], dt_bias=p["dt_bias"], dt_softplus=True,
            lambda_mode="positive", lambda_level_max=L, lambda_level_base=2,
            lambda_htype=HType.WEAK, lambda_hstruct=HStruct.MAMBA2, lambda_level_fixed=True)
        outs.append((out, S.states))
    assert outs[0][0].dtype == F32
    for a, b in zip(*outs):
        assert torch.equal(a, b)
