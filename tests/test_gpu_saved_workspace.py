"""The forward workspace that a training call holds for its backward is one of the node's
saved tensors: saved-tensor hooks (offloading, for instance) see it, and it goes when the
backward has run, also while the output is still referred to."""
import gc

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _call(kind):
    """(function, leaves): a training call long enough that it holds a workspace."""
    from hattention.base import HStruct, HType
    from hattention.kernel import hattention_kernel
    from hattention.mamba_apis import hmamba_chunk_scan_combined, hmamba_split_conv1d_scan_combined
    gen = torch.Generator(DEV).manual_seed(5)
    rn = lambda *s, dtype=torch.bfloat16: torch.randn(*s, device=DEV, generator=gen).to(dtype)
    B, S, H, P, N, L = 1, 2048, 2, 64, 64, 12
    neg = lambda *s: -torch.rand(*s, device=DEV, generator=gen)
    kw = dict(lambda_mode="positive", lambda_level_max=L, lambda_level_base=2,
              lambda_htype=HType.WEAK, lambda_hstruct=HStruct.MAMBA2, lambda_level_fixed=True)
    if kind.startswith("gdn"):
        V = int(kind[3:])
        xs = [rn(B, S, H, N), rn(B, S, H, N), rn(B, S, H, V), torch.sigmoid(rn(B, S, H)),
              0.05 * neg(B, S, H), torch.sigmoid(rn(B, S, H, L))]
        fn = lambda q, k, v, b, g, l: hattention_kernel(
            q, k, v, b, g, l, 0.125, False, 2, HType.WEAK, HStruct.GDELTA,
            use_qk_l2norm_in_kernel=True)
    elif kind == "scan":
        xs = [rn(B, S, H, P), rn(B, S, H), neg(H), rn(B, S, 1, N), rn(B, S, 1, N),
              rn(B, S, H, L), rn(H, L), rn(H), rn(H)]
        fn = lambda x, dt, A, Bm, Cm, dl, Lp, D, db: hmamba_chunk_scan_combined(
            x, dt, A, Bm, Cm, dl, Lp, 64, D=D, dt_bias=db, dt_softplus=True, **kw)[0]
    else:
        dim, c = H * P, H * P + 2 * N
        xs = [rn(B, S, dim + c + H + H * L), rn(c, 4), rn(c), rn(H), neg(H), rn(H, L), rn(H),
              rn(dim), rn(dim, dim)]
        fn = lambda z, cw, cb, db, A, Lp, D, rw, ow: hmamba_split_conv1d_scan_combined(
            z, cw, cb, db, A, Lp, D, 64, rmsnorm_weight=rw, rmsnorm_eps=1e-6, outproj_weight=ow,
            headdim=P, ngroups=1, norm_before_gate=False, **kw)
    return fn, [x.requires_grad_() for x in xs]


@pytest.mark.parametrize("kind", ["gdn64", "gdn192", "scan", "split"])
def test_workspace_is_a_saved_tensor(kind):
    print(f"[saved workspace] {kind}", flush=True)
    fn, xs = _call(kind)
    gc.collect()             # (nothing of earlier calls goes while memory is counted)
    torch.cuda.synchronize()

    def step(hooks):
        base = torch.cuda.memory_allocated()
        if hooks:
            with torch.autograd.graph.save_on_cpu():
                o = fn(*xs)
        else:
            o = fn(*xs)
        held = torch.cuda.memory_allocated() - base
        # (retained, then again: what the first backward read is whole for the second)
        g1 = torch.autograd.grad(o, xs, torch.ones_like(o), retain_graph=True)
        g2 = torch.autograd.grad(o, xs, torch.ones_like(o))
        assert all(torch.equal(a, b) for a, b in zip(g1, g2))
        del g2
        after = torch.cuda.memory_allocated() - base - sum(-(-g.nbytes // 512) * 512 for g in g1)
        return o, g1, held, after

    step(False)              # (what libraries allocate at their first call)
    o, ref, held, after = step(False)
    out = -(-o.nbytes // 512) * 512
    assert held > out and after <= out
    del o
    o, got, held, _ = step(True)
    assert held <= out       # all of it moved to the host
    assert all(torch.equal(a, b) for a, b in zip(ref, got))
