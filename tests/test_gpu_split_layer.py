"""HMambaSplitFunction (the split-conv layer as one autograd node) against the chain of
its parts, CausalConv1dSilu -> HMambaScanFunction -> GatedRMSNorm: the same bits in the
output and in every gradient, for parameters in bf16 and fp32, grouped B / C, and where
the folded scan does not apply (fp32 activations, headdim 128 without its summaries).
What both sides share, the kernels and the scan's forward and backward, is compared with
the oracle in test_gpu_mamba_layer.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("B,S,H,P,G,act,par,bias", [
    (2, 128, 3, 64, 1, torch.bfloat16, torch.bfloat16, True),
    (1, 1088, 4, 64, 2, torch.bfloat16, torch.float32, True),
    (1, 64, 2, 128, 2, torch.bfloat16, torch.bfloat16, False),
    (1, 192, 2, 64, 1, torch.float32, torch.float32, True)])
def test_one_node_equals_the_chain(B, S, H, P, G, act, par, bias):
    from hattention.base import HStruct, HType
    from hattention.mamba_apis import hmamba_chunk_scan_combined, hmamba_split_conv1d_scan_combined
    from hattention.mamba_layer import CausalConv1dSilu, GatedRMSNorm
    N, L, W = 64, 7 + max(0, (S // 64 - 1).bit_length()), 4
    dim, gn = H * P, G * N
    print(f"[split node] B={B} S={S} H={H} P={P} G={G} {act} {par}", flush=True)
    gen = torch.Generator(DEV).manual_seed(S)
    rn = lambda *s, dtype=par: torch.randn(*s, device=DEV, generator=gen).to(dtype)
    base = dict(z=rn(B, S, 2 * dim + 2 * gn + H + H * L, dtype=act), cw=rn(dim + 2 * gn, W),
                cb=rn(dim + 2 * gn) if bias else None, db=rn(H), A=-torch.rand(H, device=DEV, generator=gen),
                L=rn(H, L), D=rn(H), rw=rn(dim), ow=rn(dim, dim) / dim ** 0.5)
    kw = dict(lambda_mode="positive", lambda_level_max=L, lambda_level_base=2,
              lambda_htype=HType.WEAK, lambda_hstruct=HStruct.MAMBA2, lambda_level_fixed=True)

    def node(p):
        return hmamba_split_conv1d_scan_combined(
            p["z"], p["cw"], p["cb"], p["db"], p["A"], p["L"], p["D"], 64, rmsnorm_weight=p["rw"],
            rmsnorm_eps=1e-6, outproj_weight=p["ow"], headdim=P, ngroups=G, norm_before_gate=False, **kw)

    def chain(p):
        x, Bm, Cm = CausalConv1dSilu.apply(p["z"], dim, dim + 2 * gn, dim, dim + gn, p["cw"], p["cb"])
        c = 2 * dim + 2 * gn
        y, _ = hmamba_chunk_scan_combined(
            x.view(B, S, H, P), p["z"][..., c:c + H], p["A"], Bm.view(B, S, G, N),
            Cm.view(B, S, G, N), p["z"][..., c + H:].reshape(B, S, H, L), p["L"], 64, D=p["D"],
            dt_bias=p["db"], dt_softplus=True, **kw)
        y = GatedRMSNorm.apply(y.reshape(B, S, dim), p["z"], 0, p["rw"], 1e-6)
        return torch.nn.functional.linear(y.to(p["ow"].dtype), p["ow"])

    res = []
    for fn in (node, chain):
        p = {n: t.clone().requires_grad_(True) if t is not None else None for n, t in base.items()}
        o = fn(p)
        dy = torch.randn(o.shape, device=DEV, generator=torch.Generator(DEV).manual_seed(7)).to(o.dtype)
        names = [n for n in p if p[n] is not None]
        res.append([o] + list(torch.autograd.grad(o, [p[n] for n in names], dy)))
    for n, a, r in zip(["o"] + names, *res):
        assert a.dtype == r.dtype and torch.equal(a, r), (n, (a.float() - r.float()).abs().max().item())
