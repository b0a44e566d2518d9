"""The multi-token state kernel (hattn_hstate_steps) against the recurrent form in
float64 on the CPU, at the edges of its lane and row blocks: level counts that
divide no lane width, K and V that leave a block part empty, every lane width the
launch chooses between (by the number of rows), cascades as deep as the state,
and more tokens than one launch takes.

Tolerances: fp32 operands 1e-5 on the output and every level (fp32 sums of at
most 256 terms: 256 eps = 3e-5 worst case, eps sqrt(256) = 2e-6 expected), bf16
1e-2 (the output's rounding).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _reference(S, depth, q, k, v, g, l, beta, strong):
    """One token on fp64 states [B, H, K, V, L]."""
    S = S.clone()
    L = S.shape[-1]
    if strong:
        old = S.clone()
        S[..., 0] = 0
        for e in range(1, min(depth + 1, L)):
            S[..., e] = old[..., e - 1] + (old[..., e] if e == depth else 0)
    elif depth:
        S[..., depth] += S[..., :depth].sum(-1)
        S[..., :depth] = 0
    S *= torch.exp(g)[..., None, None, None]
    if beta is not None:
        kS = torch.einsum("bhk,bhkvl->bhvl", k, S)
        S -= (beta[..., None] * k)[..., None, None] * kS[:, :, None]
        v = v * beta[..., None]
    S[..., 0] = k[..., None] * v[:, :, None]
    return torch.einsum("bhk,bhkvl,bhl->bhv", q, S, l), S


CASES = [  # B, H, K, V, L, T
    (1, 1, 64, 16, 5, 16), (1, 2, 17, 48, 7, 64), (2, 3, 100, 32, 18, 9), (1, 1, 256, 16, 32, 5),
    (24, 16, 64, 64, 18, 3), (40, 16, 33, 128, 14, 2), (8, 16, 128, 128, 19, 3), (1, 1, 64, 16, 1, 1),
    (1, 2, 64, 16, 3, 4), (1, 1, 16, 16, 10, 300), (16, 16, 192, 48, 11, 6),
    # the widest lanes at the most rows, where the operands nearly fill the LDS
    (4, 16, 256, 64, 11, 6), (4, 16, 225, 64, 11, 5)]


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("gdn", [False, True])
@pytest.mark.parametrize("B,H,K,V,L,T", CASES)
def test_steps_match_recurrent(B, H, K, V, L, T, gdn, strong):
    from hattention.base import HStruct, HType
    from hattention.recurrent import HState, launch_step, launch_steps
    htype = HType.STRONG if strong else HType.WEAK
    print(f"[steps] B={B} H={H} K={K} V={V} L={L} T={T} gdn={gdn} strong={strong}", flush=True)
    gen = torch.Generator().manual_seed(L * 100 + K)
    G = 1 if H % 2 else 2
    rn = lambda *s: torch.randn(*s, generator=gen)
    q, k = rn(B, T, G, K), rn(B, T, G, K) / K ** 0.5
    v, g, l = rn(B, T, H, V), -0.1 * torch.rand(B, T, H, generator=gen), rn(B, T, H, L)
    beta = torch.rand(B, T, H, generator=gen) if gdn else None
    hs = HStruct.GDELTA if gdn else HStruct.MAMBA2
    S = HState(2, htype, hs, (B, H, K, V, L), torch.float32, DEV)
    one = HState(2, htype, hs, (B, H, K, V, L), torch.float32, DEV)
    d = {n: t.to(DEV) if t is not None else None
         for n, t in dict(q=q, k=k, v=v, beta=beta, g=g, l=l).items()}
    o = torch.empty(B, T, H, V, device=DEV)
    launch_steps(S, 0, T, o=o, **d)
    plan = HState(2, htype, hs, (1, 1, 1, 1, L), torch.float32, "cpu")
    ref, big = torch.zeros(B, H, K, V, L, dtype=torch.float64, device=DEV), T <= 20
    rep = lambda t: t.repeat_interleave(H // G, 1)
    outs = []
    for t in range(T):
        at = [x[:, t].double() if x is not None else None
              for x in (d["q"], d["k"], d["v"], d["g"], d["l"], d["beta"])]
        ot, ref = _reference(ref, plan.plan_cascade(), rep(at[0]), rep(at[1]), *at[2:], strong)
        outs.append(ot)
        if big:   # and one launch per token
            o1 = torch.empty(B, H, V, device=DEV)
            launch_step(one, q=d["q"][:, t].contiguous(), k=d["k"][:, t].contiguous(),
                        v=d["v"][:, t].contiguous(), g=d["g"][:, t].contiguous(),
                        beta=d["beta"][:, t].contiguous() if gdn else None,
                        l=d["l"][:, t].contiguous(), o=o1, update=True, output=True)
            assert torch.equal(o1, o[:, t])
    want = torch.stack(outs, 1)
    assert (o.double() - want).norm() < 1e-5 * want.norm()
    for e in range(L):
        r, x = ref[..., e], S.states[..., e].double()
        assert (x - r).norm() <= 1e-5 * r.norm(), e
    assert S.counts.tolist() == plan.host_counts == S.host_counts
    if big:
        assert torch.equal(one.states, S.states) and one.counts.tolist() == plan.host_counts


def test_steps_overflow_stops_where_the_step_does():
    """A two-level state holds 2 tokens: the third raises, the first two are stepped."""
    from hattention.base import HStruct, HType
    from hattention.recurrent import HState, launch_steps
    S = HState(2, HType.WEAK, HStruct.MAMBA2, (1, 1, 16, 16, 2), torch.float32, DEV)
    x = torch.ones(1, 5, 1, 16, device=DEV)
    n = 0
    probe = HState(2, HType.WEAK, HStruct.MAMBA2, (1, 1, 1, 1, 2), torch.float32, "cpu")
    with pytest.raises(IndexError):
        while True:
            probe.plan_cascade()
            n += 1
    with pytest.raises(IndexError):
        launch_steps(S, 0, 5, k=x, v=x, g=torch.zeros(1, 5, 1, device=DEV))
    assert S.host_counts == probe.host_counts == S.counts.tolist()
    assert S.states.sum().item() == n * 16 * 16


@pytest.mark.parametrize("offset", [1, 2])
def test_steps_on_unaligned_state(offset):
    """A state view that starts 4 or 8 bytes into its storage takes narrower loads."""
    from hattention.base import HStruct, HType
    from hattention.recurrent import HState, launch_steps
    B, H, K, V, L, T = 40, 16, 64, 64, 18, 3
    gen = torch.Generator(DEV).manual_seed(3)
    S = [HState(2, HType.WEAK, HStruct.MAMBA2, (B, H, K, V, L), torch.float32, DEV) for _ in range(2)]
    S[1].states = torch.zeros(B * H * K * V * L + 4, device=DEV)[offset:-(4 - offset)].view(B, H, K, V, L)
    x = {n: torch.randn(B, T, H, s, device=DEV, generator=gen) for n, s in (("q", K), ("k", K), ("v", V), ("l", L))}
    g = -torch.rand(B, T, H, device=DEV, generator=gen)
    o = [torch.empty(B, T, H, V, device=DEV) for _ in range(2)]
    for i in range(2):
        launch_steps(S[i], 0, T, g=g, o=o[i], **x)
    assert (o[0] - o[1]).norm() < 1e-5 * o[0].norm()
    assert (S[0].states - S[1].states).norm() < 1e-6 * S[0].states.norm()
