"""The performance cases of log-linear attention on one GPU.

Each case is one call (or one training step) that a program using this package
makes through its public entry points:

* ``scan``         hattention_kernel with HStruct.MAMBA2: the bare chunkwise scan
* ``layer``        hmamba_split_conv1d_scan_combined: a training step of the Mamba-2 layer
* ``prefill``      hmamba_chunk_scan_combined returning the HState of a prompt
* ``decode``       hselective_state_update: one token of the Mamba-2 layer
* ``gdn``          chunk_h_gated_delta_rule: the chunkwise Gated DeltaNet
* ``gdn_prefill``  chunk_h_gated_delta_rule returning the HState of a prompt
* ``gdn_decode``   chunk_h_gated_delta_rule: one token from an HState

``listed()`` holds the fixed cases, ``draw(rng)`` one more of the same ranges,
``prepare`` / ``run`` make and use a case's inputs, ``work`` gives the bytes and
operations that it cannot do without, ``exact`` the result in 64 bits by plain
torch, ``tolerance`` how far another correct implementation may be from it.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..",
                                "log-linear-attention_amd"))

from hattention.base import HStruct, HType  # noqa: E402
from hattention.gated_delta_rule_apis import chunk_h_gated_delta_rule  # noqa: E402
from hattention.kernel import hattention_kernel  # noqa: E402
from hattention.mamba_apis import (hmamba_chunk_scan_combined,  # noqa: E402
                                   hmamba_split_conv1d_scan_combined, hselective_state_update)
from hattention.recurrent import HState  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEV = "cuda:0"
CHUNK = 64
LOW = 7              # levels inside one chunk of 64 tokens
STATE_LEVELS = 18    # decode state of a 131072-token context
CONV = 4             # taps of the layer's causal convolution
DECODED = 1000       # tokens in a decode state before the call
# The layer's training step leaves the decay's parameters as they are: on random
# data their gradients are sums over all tokens in which the terms cancel, and in
# bf16 no digit of them is left to compare (their part of the input's gradient,
# ddt, is compared).
FROZEN = ("A", "dt_bias")


def _levels(T):
    """Levels of a sequence of T tokens (whole chunks)."""
    return LOW + max(0, math.ceil(math.log2(max(1, -(-T // CHUNK)))))


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # one token for one user of the Mamba-2 layer: nothing but latency
        dict(name="decode_one", kind="decode", B=1, H=16, P=64, N=64, G=1),
        # one token for a small batch of a Gated DeltaNet layer
        dict(name="gdn_decode", kind="gdn_decode", B=4, H=16, K=128, V=128),
        # a short training step of the bare scan: small models, fine-tuning on short texts
        dict(name="scan_train_short", kind="scan", B=2, T=1024, G=4, H=4, K=64, V=64, dtype="bf16",
             strong=False, train=True),
        # evaluation of long sequences in the training shape
        dict(name="scan_fwd", kind="scan", B=4, T=16384, G=16, H=16, K=64, V=64, dtype="bf16",
             strong=False, train=False),
        # a long context in full precision, values twice as wide as keys
        dict(name="scan_fwd_fp32", kind="scan", B=1, T=32768, G=32, H=32, K=64, V=128,
             dtype="fp32", strong=False, train=False),
        # the training step of the bare scan, 24 heads
        dict(name="scan_train", kind="scan", B=8, T=8192, G=24, H=24, K=64, V=64, dtype="bf16",
             strong=False, train=True),
        # the same with the strong hierarchy
        dict(name="strong_train", kind="scan", B=4, T=8192, G=16, H=16, K=64, V=64, dtype="bf16",
             strong=True, train=True),
        # the training step of a whole Mamba-2 layer, all parameters in bf16
        dict(name="layer_train", kind="layer", B=4, T=16384, H=16, P=64, N=64, G=1, params="bf16"),
        # a prompt whose length is no multiple of the chunk, ready for decoding
        dict(name="prefill", kind="prefill", B=2, T=4005, H=16, P=64, N=64, G=1),
        # the training step of a Gated DeltaNet layer, heads of 128
        dict(name="gdn_train", kind="gdn", B=4, T=8192, G=16, H=16, K=128, V=128, dtype="bf16",
             train=True),
        # and of the model configuration with six heads of 192, values twice as wide
        dict(name="gdn_train_wide", kind="gdn", B=1, T=16384, G=6, H=6, K=192, V=384,
             dtype="bf16", train=True),
        # a prompt of a Gated DeltaNet layer, ready for decoding
        dict(name="gdn_prefill", kind="gdn_prefill", B=1, T=2085, H=16, K=128, V=128),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _group(rng, H):
    """Key / query heads: one per head, one for all, or a divisor between."""
    return rng.choice([H, 1, rng.choice([g for g in range(1, H + 1) if H % g == 0])])


_COST = {  # the most that a drawn case of each kind may take: bytes, operations
    "scan": (1.72e9, 2.8e11), "layer": (9.2e8, 6.2e11), "prefill": (3e8, 2e11),
    "decode": (4e8, 1e9), "gdn": (1.2e9, 9.4e11), "gdn_prefill": (3e8, 3e11),
    "gdn_decode": (4e8, 1e9)}


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "layer", "prefill", "decode", "gdn", "gdn",
                       "gdn_prefill", "gdn_decode"])
    while True:
        H = _log(rng, 1, 32)
        if kind == "scan":
            strong, train = rng.random() < 0.25, rng.random() < 0.6
            c = dict(kind=kind, B=_log(rng, 1, 8), T=CHUNK * _log(rng, 1, 128 if train else 512),
                     G=_group(rng, H), H=H, K=64 if strong else rng.choice([64, 64, 64, 128]),
                     V=64 if strong else rng.choice([64, 64, 64, 128]),
                     dtype="bf16" if strong else rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]),
                     strong=strong, train=train)
        elif kind == "layer":
            c = dict(kind=kind, B=_log(rng, 1, 4), T=CHUNK * _log(rng, 2, 256), H=H, P=64, N=64,
                     G=_group(rng, H), params=rng.choice(["bf16", "bf16", "fp32"]))
        elif kind == "prefill":
            c = dict(kind=kind, B=_log(rng, 1, 8), T=_log(rng, 16, 8192), H=H, P=64, N=64,
                     G=_group(rng, H))
        elif kind == "decode":
            c = dict(kind=kind, B=_log(rng, 1, 64), H=H, P=64, N=64, G=_group(rng, H))
        else:
            H = _log(rng, 1, 16)
            c = dict(kind=kind, B=_log(rng, 1, 4), H=H, K=rng.choice([64, 128, 128, 192, 256]),
                     V=rng.choice([64, 128, 128, 256, 384]))
            if kind == "gdn":
                c.update(T=CHUNK * _log(rng, 1, 256), G=_group(rng, H),
                         dtype=rng.choice(["bf16", "bf16", "fp16"]), train=rng.random() < 0.7)
            elif kind == "gdn_prefill":
                c.update(T=_log(rng, 65, 4096))
            else:
                c.update(B=_log(rng, 1, 32))
        w = work(c)
        if w["bytes"] <= _COST[kind][0] and w["flops"] <= _COST[kind][1]:
            return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
class _Make:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(DEV).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, scale=1.0, shift=0.0):
        x = torch.randn(*shape, generator=self.gen, device=DEV)
        return (x * scale + shift).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.gen, device=DEV) * (hi - lo) + lo

    def decay(self, B, T, H):
        """The log-decays of a Mamba-2 layer at its initialisation: -A dt, A from 1
        to 16 and dt from 0.001 to 0.1, both spread over their logarithm by head."""
        A = torch.exp(self.uniform(H, lo=0.0, hi=math.log(16.0)))
        dt0 = torch.exp(self.uniform(H, lo=math.log(1e-3), hi=math.log(1e-1)))
        bias = dt0 + torch.log(-torch.expm1(-dt0))
        dt = torch.nn.functional.softplus(self.normal(B, T, H) + bias).clamp(1e-3, 1e-1)
        return -A * dt

    def weights(self, *shape, dtype):
        """Level weights lambda."""
        return torch.nn.functional.softplus(self.normal(*shape)).to(dtype)


def _mamba(c, m, pdt):
    """Per-head parameters of a Mamba-2 layer."""
    H = c["H"]
    dt0 = torch.exp(m.uniform(H, lo=math.log(1e-3), hi=math.log(1e-1)))
    return dict(A=-torch.exp(m.uniform(H, lo=0.0, hi=math.log(16.0))),
                dt_bias=(dt0 + torch.log(-torch.expm1(-dt0))).to(pdt),
                D=m.normal(H, dtype=pdt, scale=0.1, shift=1.0))


def _lambda_opts(L):
    return dict(lambda_mode="positive", lambda_level_max=L, lambda_level_base=2,
                lambda_htype=HType.WEAK, lambda_hstruct=HStruct.MAMBA2, lambda_level_fixed=True)


def _decode_state(m, B, H, K, V, hstruct):
    """The HState after DECODED tokens: level 0 holds the last token, level e >= 1
    holds 2^(e-1) tokens where bit e - 1 of the earlier tokens' number is set."""
    S = HState(2, HType.WEAK, hstruct, (B, H, K, V, STATE_LEVELS), torch.float32, DEV)
    counts = [1] + [2 ** e if (DECODED - 1) >> e & 1 else 0 for e in range(STATE_LEVELS - 1)]
    for e, n in enumerate(counts):
        if n:
            S.states[..., e] = m.normal(B, H, K, V, scale=min(n, 32) ** 0.5)
    S.set_counts(counts)
    return S


def prepare(case, seed):
    c, m, bf = case, _Make(seed), torch.bfloat16
    kind, B, H = c["kind"], c["B"], c["H"]
    s = dict(case=dict(c))
    if kind in ("scan", "gdn"):
        T, G, K, V, dt = c["T"], c["G"], c["K"], c["V"], DTYPES[c["dtype"]]
        L = _levels(T)
        s["x"] = dict(q=m.normal(B, T, G, K, dtype=dt), k=m.normal(B, T, G, K, dtype=dt),
                      v=m.normal(B, T, H, V, dtype=dt), g=m.decay(B, T, H),
                      l=m.weights(B, T, H, L, dtype=dt))
        if kind == "gdn":
            s["x"]["beta"] = torch.sigmoid(m.normal(B, T, H)).to(dt)
        s["do"] = m.normal(B, T, H, V, dtype=dt) if c["train"] else None
    elif kind == "layer":
        T, P, N, G, pdt = c["T"], c["P"], c["N"], c["G"], DTYPES[c["params"]]
        L, dim, gn = _levels(T), H * P, G * N
        z = m.normal(B, T, 2 * dim + 2 * gn + H + H * L)
        z[..., 2 * dim + 2 * gn:2 * dim + 2 * gn + H] *= 0.5
        s["x"] = dict(z=z.to(bf), conv_w=m.normal(dim + 2 * gn, CONV, dtype=pdt, scale=0.5),
                      conv_b=m.normal(dim + 2 * gn, dtype=pdt, scale=0.1), **_mamba(c, m, pdt),
                      L=m.normal(H, L, dtype=pdt, scale=0.5),
                      norm_w=m.normal(dim, dtype=pdt, scale=0.1, shift=1.0),
                      out_w=m.normal(dim, dim, dtype=pdt, scale=dim ** -0.5),
                      out_b=m.normal(dim, dtype=pdt, scale=0.1))
        s["do"] = m.normal(B, T, dim, dtype=pdt)
    elif kind in ("prefill", "decode"):
        P, N, G = c["P"], c["N"], c["G"]
        L = STATE_LEVELS
        lead = (B, c["T"]) if kind == "prefill" else (B,)
        s["x"] = dict(x=m.normal(*lead, H, P, dtype=bf), dt=m.normal(*lead, H, dtype=bf, scale=0.5),
                      Bm=m.normal(*lead, G, N, dtype=bf), Cm=m.normal(*lead, G, N, dtype=bf),
                      dl=m.normal(*lead, H, L, dtype=bf), L=m.normal(H, L, dtype=bf, scale=0.5),
                      **_mamba(c, m, bf))
        if kind == "decode":
            s["state"] = _decode_state(m, B, H, N, P, HStruct.MAMBA2)
    else:
        T, K, V = c.get("T", 1), c["K"], c["V"]
        s["x"] = dict(q=m.normal(B, T, H, K, dtype=bf), k=m.normal(B, T, H, K, dtype=bf),
                      v=m.normal(B, T, H, V, dtype=bf), g=m.decay(B, T, H),
                      l=m.weights(B, T, H, STATE_LEVELS, dtype=bf),
                      beta=torch.sigmoid(m.normal(B, T, H)).to(bf))
        if kind == "gdn_decode":
            s["state"] = _decode_state(m, B, H, K, V, HStruct.GDELTA)
    if s.get("do") is not None:
        for n, t in s["x"].items():
            t.requires_grad_(n not in FROZEN)
    return s


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _scan(x, strong):
    return hattention_kernel(x["q"], x["k"], x["v"], None, x["g"], x["l"], None, False, 2,
                             HType.STRONG if strong else HType.WEAK, HStruct.MAMBA2)


def _layer(x, c):
    return hmamba_split_conv1d_scan_combined(
        x["z"], x["conv_w"], x["conv_b"], x["dt_bias"], x["A"], x["L"], x["D"], CHUNK,
        rmsnorm_weight=x["norm_w"], rmsnorm_eps=1e-6, outproj_weight=x["out_w"],
        outproj_bias=x["out_b"], headdim=c["P"], ngroups=c["G"], norm_before_gate=False,
        **_lambda_opts(x["L"].shape[-1]))


def _gdn(x, **kw):
    return chunk_h_gated_delta_rule(x["q"], x["k"], x["v"], x["g"], x["l"], x["beta"],
                                    use_qk_l2norm_in_kernel=True, **kw)


def run(state):
    c, x = state["case"], state["x"]
    kind = c["kind"]
    if kind in ("scan", "layer", "gdn"):
        def call():
            if kind == "scan":
                return _scan(x, c["strong"])
            return _layer(x, c) if kind == "layer" else _gdn(x)[0]
        if state["do"] is None:
            with torch.no_grad():
                return {"o": call()}
        o = call()
        names = [n for n in x if x[n].requires_grad]
        grads = torch.autograd.grad(o, [x[n] for n in names], state["do"])
        return {"o": o, **{"d" + n: t for n, t in zip(names, grads)}}
    if kind == "prefill":
        y, S = hmamba_chunk_scan_combined(
            x["x"], x["dt"], x["A"], x["Bm"], x["Cm"], x["dl"], x["L"], CHUNK, D=x["D"],
            dt_bias=x["dt_bias"], dt_softplus=True, return_final_states=True,
            **_lambda_opts(STATE_LEVELS))
    elif kind == "decode":
        y, S = hselective_state_update(
            state["state"], x["x"], x["dt"], x["A"], x["Bm"], x["Cm"], x["dl"], x["L"], D=x["D"],
            dt_bias=x["dt_bias"], dt_softplus=True, **_lambda_opts(STATE_LEVELS))
    else:
        with torch.no_grad():
            y, S = _gdn(x, initial_state=state.get("state"), output_final_state=True)
    return {"o": y, "states": S.states, "counts": S.counts}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _scan_flops(B, T, H, K, V, train):
    """Causal 64 x 64 tiles and their products, each chunk's state update, and
    the reads of the inter-chunk levels (half of them per chunk)."""
    lev = _levels(T) - LOW
    f = 2 * T * CHUNK * (K + V) + 2 * T * K * V + T * K * V * lev
    if train:
        f += 2 * T * CHUNK * (3 * K + 2 * V) + 6 * T * K * V + 2 * T * K * V * lev
    return B * H * f


def _gdn_flops(B, T, H, K, V, train):
    """Chunk products (K K^T, Q K^T, W, q_new, U, A V), the triangular inverse, and
    per level the delta-rule step and the read; the backward twice that again."""
    lev = _levels(T) - LOW
    f = 2 * T * CHUNK * (5 * K + 2 * V + CHUNK) + 2 / 3 * CHUNK * CHUNK * T + 5 * T * K * V * lev
    return B * H * f * (3 if train else 1)


def work(case):
    c = case
    kind, B, H = c["kind"], c["B"], c["H"]
    if kind in ("scan", "gdn"):
        T, G, K, V, e = c["T"], c["G"], c["K"], c["V"], DTYPES[c["dtype"]].itemsize
        L = _levels(T)
        ins = 2 * G * K * e + H * V * e + H * 4 + H * L * e + (H * e if kind == "gdn" else 0)
        per = ins + H * V * e
        if c["train"]:
            per += ins + H * V * e      # the gradients, and dO
        f = (_scan_flops if kind == "scan" else _gdn_flops)(B, T, H, K, V, c["train"])
        return {"bytes": B * T * per, "flops": f}
    if kind == "layer":
        T, P, N, G = c["T"], c["P"], c["N"], c["G"]
        dim, L, pe = H * P, _levels(T), DTYPES[c["params"]].itemsize
        Z = 2 * dim + 2 * G * N + H + H * L
        nbytes = B * T * (2 * 2 * Z + 2 * pe * dim) + 2 * pe * dim * dim
        f = _scan_flops(B, T, H, N, P, True) + 6 * B * T * dim * dim + \
            B * T * (dim + 2 * G * N) * CONV * 6
        return {"bytes": nbytes, "flops": f}
    if kind in ("decode", "prefill"):
        K, V, G = c["N"], c["P"], c["G"]
        io = 2 * (2 * H * V + 2 * G * K + H + H * STATE_LEVELS)
    else:
        K, V = c["K"], c["V"]
        io = 2 * H * (2 * K + 2 * V + STATE_LEVELS + 1) + 4 * H
    states = B * H * K * V * STATE_LEVELS
    if kind in ("decode", "gdn_decode"):
        per = 5 if kind == "decode" else 9
        return {"bytes": 2 * 4 * states + B * io, "flops": per * states}
    T = c["T"]
    f = (_scan_flops if kind == "prefill" else _gdn_flops)(B, T, H, K, V, False)
    return {"bytes": B * T * io + 4 * states, "flops": f}


# --------------------------------------------------------------------------
# tolerances
# --------------------------------------------------------------------------
def tolerance(case):
    """About four times the largest error against ``exact`` seen over these ranges,
    over all outputs of the case: in the scan's training steps that is dg, the sum
    over all later tokens of differences q . dq - k . dk whose terms cancel
    (bf16 0.005 to 0.026, growing with T, where every other output is at 0.003), and
    "max" is about four times the largest single difference."""
    kind, dtype, train = case["kind"], case.get("dtype", "bf16"), case.get("train", True)
    if kind == "scan":
        rel, most = {"bf16": (0.03, 0.8) if train else (0.01, 0.2),
                     "fp16": (7e-3, 0.03) if train else (1.5e-3, 0.015),
                     "fp32": (1.3e-4, 1e-3) if train else (3e-5, 7e-4)}[dtype]
    elif kind == "gdn":
        rel, most = {"bf16": (0.02, 0.5), "fp16": (8e-3, 0.2)}[dtype]
    else:
        rel, most = {"layer": (0.015, 0.9), "prefill": (0.01, 0.3), "decode": (0.012, 0.06),
                     "gdn_decode": (0.012, 0.06), "gdn_prefill": (0.02, 0.4)}[kind]
    return {"rel": rel, "max": most}


# --------------------------------------------------------------------------
# the results in 64 bits
# --------------------------------------------------------------------------
def _head_first(t, H=None):
    """[B, T, G, ...] -> [B, H, T, ...], groups repeated per head."""
    t = t.transpose(1, 2)
    return t if H is None or t.shape[1] == H else t.repeat_interleave(H // t.shape[1], dim=1)


def _weak_scan(q, k, v, g, l):
    """o_t = sum_{s <= t} l[t, bit_length(t ^ s)] exp(G_t - G_s) (q_t . k_s) v_s, all
    [B, H, T, .]: level e pairs the two halves of each block of 2^e tokens."""
    B, H, T, K = q.shape
    V = v.shape[-1]
    top = max(0, math.ceil(math.log2(T)))
    pad = 2 ** top - T
    fill = lambda t: torch.nn.functional.pad(t, (0, 0, 0, pad))  # noqa: E731
    q, k, v, l, Gc = fill(q), fill(k), fill(v), fill(l), torch.cumsum(fill(g[..., None]), 2)
    o = l[..., :1] * (q * k).sum(-1, keepdim=True) * v
    for e in range(1, top + 1):
        h = 2 ** (e - 1)
        half = lambda t, i: t.reshape(B, H, -1, 2, h, t.shape[-1])[:, :, :, i]  # noqa: E731
        mid = half(Gc, 0)[..., -1:, :]
        qe, ke, ve = half(q, 1), half(k, 0) * torch.exp(mid - half(Gc, 0)), half(v, 0)
        oe = (qe @ ke.transpose(-1, -2)) @ ve if h <= CHUNK else qe @ (ke.transpose(-1, -2) @ ve)
        oe = oe * torch.exp(half(Gc, 1) - mid) * half(l[..., e:e + 1], 1)
        o = o + torch.stack([torch.zeros_like(oe), oe], 3).reshape(B, H, -1, V)
    return o[:, :, :T]


def _strong_levels(n):
    """The strong level of every pair t > s below n (0 elsewhere): with 2^a the
    largest power of two up to t and u = 2^max(a-1, 0), sources below u, and those
    below 2u for targets from 2^a + u, are at level a + 1; the others are pairs
    of the same hierarchy u (sources below 2u) or 2u tokens further left."""
    t = torch.arange(n)[:, None].expand(n, n).clone()
    s = torch.arange(n)[None].expand(n, n).clone()
    out, live = torch.zeros(n, n, dtype=torch.long), s < t
    while bool(live.any()):
        a = torch.frexp(t.clamp(min=1).double())[1].long() - 1
        u = 2 ** (a - 1).clamp(min=0)
        done = live & ((s < u) | ((s < 2 * u) & (t - 2 ** a >= u)))
        out[done] = a[done] + 1
        live &= ~done
        step = torch.where(s < 2 * u, u, 2 * u) * live
        t, s = t - step, s - step
    return out


def _strong_scan(q, k, v, g, l):
    """The same sum with the strong level of each pair: one table for pairs within
    a chunk, one for neighbouring chunks, one level for pairs of farther chunks."""
    B, H, T, K = q.shape
    N = T // CHUNK
    ch = lambda t: t.reshape(B, H, N, CHUNK, t.shape[-1])  # noqa: E731
    q, k, v, l = ch(q), ch(k), ch(v), ch(l)
    Gc = torch.cumsum(ch(g[..., None]), 3)
    last = Gc[..., -1:, :]
    near = _strong_levels(2 * CHUNK).to(q.device)
    pick = lambda t, tab: torch.gather(t, -1, tab.expand(*t.shape[:3], CHUNK, CHUNK))  # noqa: E731
    lower = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    dec = torch.exp((Gc - Gc.transpose(-1, -2)).masked_fill(~lower, -math.inf))
    o = ((q @ k.transpose(-1, -2)) * dec * pick(l, near[:CHUNK, :CHUNK])) @ v
    kd = k * torch.exp(last - Gc)
    if N > 1:
        S = (q[:, :, 1:] * torch.exp(Gc[:, :, 1:])) @ kd[:, :, :-1].transpose(-1, -2)
        sub = (S * pick(l[:, :, 1:], near[CHUNK:, :CHUNK])) @ v[:, :, :-1]
        o = o + torch.cat([torch.zeros_like(o[:, :, :1]), sub], 2)
    if N > 2:
        far = _strong_levels(N).to(q.device).tril(-2)
        kv = (kd.transpose(-1, -2) @ v).flatten(3)
        E = torch.cumsum(last[..., 0, 0], -1)
        before = torch.nn.functional.pad(E, (1, 0))[..., :-1]      # decay up to a chunk's start
        gap = before[..., :, None] - E[..., None, :]
        for j in range(2, int(far.max()) + 1):
            W = torch.exp(gap.masked_fill(far != j, -math.inf))
            st = (W @ kv).reshape(B, H, N, K, -1)
            o = o + (q @ st) * torch.exp(Gc) * l[..., 5 + j + 1:5 + j + 2]
    return o.reshape(B, H, T, -1)


def _unit(t):
    return t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6)


def _delta_scan(q, k, v, g, l, beta):
    """The chunkwise Gated DeltaNet, all [B, H, T, .]: in a chunk the gated
    products of I - beta k k^T by the inverse of I + A, A[r, s] = beta_r k_r . k_s
    for r > s; between chunks one state per level, moved on by each chunk's whole
    transition, written while the level's block is in its first half and read in
    its second."""
    B, H, T, K = q.shape
    N = T // CHUNK
    ch = lambda t: t.reshape(B, H, N, CHUNK, t.shape[-1])  # noqa: E731
    q, k, v, l = ch(_unit(q)), ch(_unit(k)), ch(v), ch(l)
    beta, Gc = ch(beta[..., None]), torch.cumsum(ch(g[..., None]), 3)
    last, kT = Gc[..., -1:, :], k.transpose(-1, -2)
    eye = torch.eye(CHUNK, dtype=q.dtype, device=q.device)
    inv = torch.linalg.solve_triangular(eye + (beta * (k @ kT)).tril(-1),
                                        eye.expand(B, H, N, CHUNK, CHUNK), upper=False)
    Tb = inv * beta.transpose(-1, -2)
    Mt = (q @ kT).tril() @ Tb
    lower = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    dec = torch.exp((Gc - Gc.transpose(-1, -2)).masked_fill(~lower, -math.inf))
    i = torch.arange(CHUNK, device=q.device)
    lev = torch.frexp((i[:, None] ^ i[None]).double())[1].long()
    w = torch.gather(l, -1, lev.expand(B, H, N, CHUNK, CHUNK))
    o = (Mt * dec * w) @ v
    qn = torch.exp(Gc) * (q - Mt @ k)
    move = torch.exp(last) * (torch.eye(K, dtype=q.dtype, device=q.device) - kT @ (Tb @ k))
    put = kT @ ((Tb * torch.exp(last - Gc).transpose(-1, -2)) @ v)
    E = l.shape[-1] - LOW
    h, far = [None] * E, []
    for n in range(N):
        acc = torch.zeros_like(o[:, :, n])
        for e in range(E):
            if n >> e & 1:
                acc = acc + l[:, :, n, :, LOW + e, None] * (qn[:, :, n] @ h[e])
            if (n + 1) % 2 ** (e + 1) == 0:
                h[e] = None
                continue
            if n >> e & 1:
                h[e] = move[:, :, n] @ h[e]
            else:
                h[e] = put[:, :, n] if h[e] is None else move[:, :, n] @ h[e] + put[:, :, n]
        far.append(acc)
    return (o + torch.stack(far, 2)).reshape(B, H, T, -1)


def _by_batch(fn, c, x, do):
    """{"o": fn(x), "d...": gradients}, a batch at a time; what has no batch is summed."""
    outs = []
    for b in range(c["B"]):
        xb = {n: (t[b:b + 1] if t.dim() > 2 else t).detach().double() for n, t in x.items()}
        names = [n for n in xb if do is not None and n not in FROZEN]
        for n in names:
            xb[n].requires_grad_(True)
        with torch.set_grad_enabled(do is not None):
            o = fn(xb)
        r = {"o": o.detach()}
        if do is not None:
            g = torch.autograd.grad(o, [xb[n] for n in names], do[b:b + 1].double())
            r.update({"d" + n: t for n, t in zip(names, g)})
        outs.append(r)
    return {n: torch.cat([r[n] for r in outs]) if n == "o" or x[n[1:]].dim() > 2
            else sum(r[n] for r in outs) for n in outs[0]}


def _mamba_inputs(x):
    """dt, g and lambda of a Mamba-2 layer ([B, T, H, .])."""
    sp = torch.nn.functional.softplus
    dt = sp(x["dt"] + x["dt_bias"])
    return dt, dt * x["A"], sp(x["L"] * x["dl"])


def _exact_layer(x, c):
    H, P, N, G, L = c["H"], c["P"], c["N"], c["G"], x["L"].shape[-1]
    dim, gn = H * P, G * N
    z, xBC, dt, dl = torch.split(x["z"], [dim, dim + 2 * gn, H, H * L], -1)
    B, T, _ = z.shape
    pad = torch.nn.functional.pad(xBC, (0, 0, CONV - 1, 0))
    pre = x["conv_b"] + sum(pad[:, j:j + T] * x["conv_w"][:, j] for j in range(CONV))
    xs, Bm, Cm = torch.split(torch.nn.functional.silu(pre), [dim, gn, gn], -1)
    xs = xs.reshape(B, T, H, P)
    dt, g, lam = _mamba_inputs(dict(x, dt=dt, dl=dl.reshape(B, T, H, L)))
    o = _weak_scan(_head_first(Cm.reshape(B, T, G, N), H), _head_first(Bm.reshape(B, T, G, N), H),
                   _head_first(xs * dt[..., None]), g.transpose(1, 2), _head_first(lam))
    y = (o.transpose(1, 2) + xs * x["D"][:, None]).reshape(B, T, dim)
    u = y * torch.nn.functional.silu(z)
    u = u * torch.rsqrt((u * u).mean(-1, keepdim=True) + 1e-6) * x["norm_w"]
    return torch.nn.functional.linear(u, x["out_w"], x["out_b"])


def _block(T, e):
    """The tokens that level e holds after T of them, or None."""
    if e == 0:
        return T - 1, T
    if not (T - 1) >> (e - 1) & 1:
        return None
    a = (T - 1) >> e << e
    return a, a + 2 ** (e - 1)


def _token_step(S, depth, q, k, v, g, l, beta=None):
    """One token on states [B, H, K, V, L]: levels below `depth` join into it, the
    gate, the token at level 0, the read."""
    S = S.clone()
    if depth:
        S[..., depth] += S[..., :depth].sum(-1)
        S[..., :depth] = 0
    S *= torch.exp(g)[..., None, None, None]
    if beta is not None:
        kS = torch.einsum("bhk,bhkvl->bhvl", k, S)
        S -= (beta[..., None] * k)[..., None, None] * kS[:, :, None]
        v = v * beta[..., None]
    S[..., 0] += k[..., None] * v[:, :, None]
    return torch.einsum("bhk,bhkvl,bhl->bhv", q, S, l), S


def _counts(T):
    return torch.tensor([1] + [2 ** e if (T - 1) >> e & 1 else 0 for e in range(STATE_LEVELS - 1)])


def exact(case, seed):
    c = case
    kind, H = c["kind"], c["H"]
    s = prepare(c, seed)
    x, do = s["x"], s.get("do")
    if kind in ("scan", "gdn"):
        def fn(d):
            a = [_head_first(d[n], H) for n in ("q", "k", "v", "g", "l")]
            a += [_head_first(d["beta"])] if kind == "gdn" else []
            f = _delta_scan if kind == "gdn" else _strong_scan if c["strong"] else _weak_scan
            return f(*a).transpose(1, 2)    # (gdn: l / scale and q * scale, the scale cancels)
        return _by_batch(fn, c, x, do)
    if kind == "layer":
        return _by_batch(lambda d: _exact_layer(d, c), c, x, do)
    x = {n: t.double() for n, t in x.items()}
    if kind in ("prefill", "decode"):
        dt, g, lam = _mamba_inputs(x)
        v = x["x"] * dt[..., None]
        rep = lambda t: t.repeat_interleave(H // c["G"], dim=-2)  # noqa: E731
        q, k, beta = rep(x["Cm"]), rep(x["Bm"]), None
        skip = x["x"] * x["D"][:, None]
    else:
        q, k, v, g, lam, beta = _unit(x["q"]), _unit(x["k"]), x["v"], x["g"], x["l"], x["beta"]
        skip = 0.0
    if kind in ("decode", "gdn_decode"):
        if kind == "gdn_decode":
            q, k, v, g, lam, beta = (t[:, 0] for t in (q, k, v, g, lam, beta))
        depth = ((DECODED - 1) ^ DECODED).bit_length()
        o, S = _token_step(s["state"].states.double(), depth, q, k, v, g, lam, beta)
        o = o + skip
        return {"o": o[:, None] if kind == "gdn_decode" else o, "states": S, "counts": None}
    T = c["T"]
    if kind == "prefill":
        o = _weak_scan(*(_head_first(t) for t in (q, k, v, g, lam))).transpose(1, 2) + skip
        S = torch.zeros(c["B"], H, c["N"], c["P"], STATE_LEVELS, dtype=torch.float64, device=DEV)
        w = torch.exp(g.sum(1, keepdim=True) - torch.cumsum(g, 1))
        for e in range(STATE_LEVELS):
            if blk := _block(T, e):
                i = slice(*blk)
                S[..., e] = torch.einsum("bthk,bthv->bhkv", k[:, i] * w[:, i, :, None], v[:, i])
        return {"o": o, "states": S, "counts": None}
    S = torch.zeros(c["B"], H, c["K"], c["V"], STATE_LEVELS, dtype=torch.float64, device=DEV)
    outs = []
    for t in range(T):
        ot, S = _token_step(S, ((t - 1) ^ t).bit_length() if t else 0,
                            *(a[:, t] for a in (q, k, v, g, lam, beta)))
        outs.append(ot)
    return {"o": torch.stack(outs, 1), "states": S, "counts": None}
