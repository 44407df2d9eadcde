"""Performance cases of the fused-MoE expert path, through its public entry points.

Four kinds of call:

* ``layer``    ``easyinfra_amd.fused_moe``: routing, expert GEMMs, combine (and shared experts).
* ``experts``  ``HipFusedMoE.forward_ep``: the expert module behind the plugin point, on rows grouped by
  (source rank, local expert), as the expert-parallel exchange delivers them.
* ``front``    ``ops.moe_prologue`` and the router on its logits: what a block runs before its experts.
* ``gemm``     ``torch.ops.ops.hip_grouped_gemm_single``: the grouped-GEMM op point.

Shapes are those of ``easyinfra_amd.workloads`` and of the benchmark (Mixtral-8x7B, DeepSeek-V2-Lite,
the Qwen3-30B-A3B 32-expert share, the tiny fp32 Mixtral, DeepSeek-V3's router).  Activations are
N(0, 1), weights N(0, 0.02), as there.  fp8 weights are e4m3 with absmax/448 scales per output channel.
"""
from __future__ import annotations

import math
import random

import torch

from easyinfra_amd import fused_moe, ops
from easyinfra_amd.moe import HipFusedMoE
import easyinfra_amd.torch_ops  # noqa: F401  (registers hip_grouped_gemm_single)

# hidden, expert intermediate, routed experts, top-k, experts on this GPU, shared intermediate
MODELS = {
    "mixtral": dict(H=4096, I=14336, E=8, k=2, local=8, shared=0, renorm=True, routing="plain"),
    "deepseek-v2-lite": dict(H=2048, I=1408, E=64, k=6, local=64, shared=2816, renorm=False, routing="zipf"),
    "qwen3-share": dict(H=2048, I=768, E=128, k=8, local=32, shared=0, renorm=True, routing="hotcold"),
    "tiny-mixtral": dict(H=1024, I=2816, E=8, k=2, local=8, shared=0, renorm=True, routing="plain"),
}
# routers of the block front: hidden, experts, top-k, grouped sigmoid gate
FRONTS = {
    "mixtral": dict(H=4096, E=8, k=2, grouped=False),
    "qwen3": dict(H=2048, E=128, k=8, grouped=False),
    "deepseek-v3": dict(H=7168, E=256, k=8, grouped=True),
}
EPS = 1e-6
FP8_MAX = 448.0


def listed():
    return [
        # A long prompt through one Mixtral-8x7B layer: the benchmark's headline call, the largest work.
        dict(name="mixtral-prefill-8192", kind="layer", model="mixtral", tokens=8192, mode="bf16", gate="softmax"),
        # One decode step of 64 sequences on the same layer: every expert's weights for a few rows each.
        dict(name="mixtral-decode-64", kind="layer", model="mixtral", tokens=64, mode="bf16", gate="softmax"),
        # A prompt of odd length on fp8 weights and activations.
        dict(name="mixtral-w8a8-3001", kind="layer", model="mixtral", tokens=3001, mode="w8a8", gate="softmax"),
        # A decode step of an odd number of sequences on fp8 weights with bf16 activations.
        dict(name="mixtral-w8a16-61", kind="layer", model="mixtral", tokens=61, mode="w8a16", gate="softmax"),
        # A prompt through many small experts with skewed popularity and shared experts.
        dict(name="dsv2-lite-4096", kind="layer", model="deepseek-v2-lite", tokens=4096, mode="bf16", gate="softmax"),
        # A middling ragged chunk of it, routed by the DeepSeek-V3 group-limited sigmoid gate.
        dict(name="dsv2-lite-gate-777", kind="layer", model="deepseek-v2-lite", tokens=777, mode="bf16", gate="sigmoid"),
        # One GPU's quarter of Qwen3-30B-A3B's experts: a single token, the smallest call ...
        dict(name="qwen3-share-1", kind="layer", model="qwen3-share", tokens=1, mode="bf16", gate="softmax"),
        # ... a decode batch ...
        dict(name="qwen3-share-32", kind="layer", model="qwen3-share", tokens=32, mode="bf16", gate="softmax"),
        # ... and a prompt chunk of odd length.
        dict(name="qwen3-share-1999", kind="layer", model="qwen3-share", tokens=1999, mode="bf16", gate="softmax"),
        # The fp32 layer: the reference's small correctness configuration at its own precision.
        dict(name="tiny-fp32-512", kind="layer", model="tiny-mixtral", tokens=512, mode="fp32", gate="softmax"),
        # The expert module in an expert-parallel group of four: rows of four source ranks for each expert.
        dict(name="experts-ep4-4100", kind="experts", model="qwen3-share", rows=4100, ep=4, mode="bf16"),
        # What a DeepSeek-V3 block runs before its experts, for a prompt.
        dict(name="front-dsv3-4096", kind="front", model="deepseek-v3", tokens=4096),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if n > 16 and n % 2 == 0 and rng.random() < 0.5:
        n += 1   # odd sizes among them
    return max(lo, min(hi, n))


def draw(rng: random.Random):
    u = rng.random()
    if u < 0.64:
        model = rng.choice(["mixtral", "mixtral", "deepseek-v2-lite", "deepseek-v2-lite", "qwen3-share", "qwen3-share",
                            "tiny-mixtral"])
        if model == "tiny-mixtral":
            return dict(kind="layer", model=model, tokens=_log_int(rng, 1, 2048), mode="fp32", gate="softmax")
        mode = rng.choice(["bf16", "bf16", "bf16", "bf16", "w8a8", "w8a8", "w8a16", "w8a16", "precise"])
        top = {"bf16": 8192, "w8a8": 8192, "w8a16": 7000, "precise": 4096}[mode]
        gate = "sigmoid" if model == "deepseek-v2-lite" and rng.random() < 0.5 else "softmax"
        return dict(kind="layer", model=model, tokens=_log_int(rng, 1, top), mode=mode, gate=gate)
    if u < 0.78:
        model = rng.choice(["mixtral", "deepseek-v2-lite", "qwen3-share"])
        ep = {"mixtral": 8, "deepseek-v2-lite": rng.choice([2, 4]), "qwen3-share": 4}[model]
        return dict(kind="experts", model=model, rows=_log_int(rng, 4, 16384), ep=ep, mode=rng.choice(["bf16", "bf16", "w8a16"]))
    if u < 0.90:
        model = rng.choice(["mixtral", "qwen3", "deepseek-v3"])
        return dict(kind="front", model=model, tokens=_log_int(rng, 1, 8192))
    model = rng.choice(["mixtral", "deepseek-v2-lite", "qwen3-share"])
    return dict(kind="gemm", model=model, rows=_log_int(rng, 8, 8192), ep=rng.choice([1, 2]))


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(gen, shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _rows_to_fp8(x):
    """e4m3 values and the absmax/448 scale of each row."""
    amax = x.float().abs().amax(dim=-1)
    s = torch.where(amax > 0, amax / FP8_MAX, torch.ones_like(amax))
    return (x.float() / s[..., None]).to(torch.float8_e4m3fn), s


def _weights_to_fp8(w):
    q = torch.empty(w.shape, dtype=torch.float8_e4m3fn, device=w.device)
    s = torch.empty(w.shape[:-1], dtype=torch.float32, device=w.device)
    for e in range(w.shape[0]):
        q[e], s[e] = _rows_to_fp8(w[e])
    return q, s


def _popularity(m):
    """Chance of each routed expert: four hot local experts at 8 times a cold one, a quarter of the
    assignments local (the Qwen3 share)."""
    p = torch.ones(m["E"], dtype=torch.float32, device="cuda")
    p[: m["local"] // 8] = 8.0
    p[m["local"]:] = 3.0 * float(p[: m["local"]].sum()) / (m["E"] - m["local"])
    return p


def _logits(m, x, gen):
    T, E, k = x.shape[0], m["E"], m["k"]
    if m["routing"] == "hotcold":
        # the picked experts stand out by about 8; a share is sent only tokens with a pick of its own
        p = _popularity(m)
        chosen = torch.multinomial(p.expand(T, E), k, replacement=False, generator=gen)
        own = torch.multinomial(p[: m["local"]].expand(T, m["local"]), 1, replacement=False, generator=gen)
        none = (chosen >= m["local"]).all(dim=1, keepdim=True)
        chosen[:, :1] = torch.where(none, own, chosen[:, :1])
        noise = _normal(gen, (T, E), 0.5, torch.float32).clamp_(-2.0, 2.0)
        return noise.scatter_add(1, chosen, torch.full((T, k), 8.0, device="cuda"))
    logits = x.float() @ _normal(gen, (m["H"], E), 0.02, torch.float32)
    if m["routing"] == "zipf":
        rank = torch.randperm(E, generator=gen, device="cuda").float() + 1.0
        logits = logits - 1.2 * torch.log(rank)
    return logits.contiguous()


def _expert_weights(m, gen, mode, n):
    dt = torch.float32 if mode == "fp32" else torch.bfloat16
    w_gu = _normal(gen, (n, 2 * m["I"], m["H"]), 0.02, dt)
    w_d = _normal(gen, (n, m["H"], m["I"]), 0.02, dt)
    if mode in ("w8a8", "w8a16"):
        (w_gu, s_gu), (w_d, s_d) = _weights_to_fp8(w_gu), _weights_to_fp8(w_d)
        return w_gu, w_d, (s_gu, s_d)
    return w_gu, w_d, None


def _counts(rows, ep, local, gen):
    """Rows per (source rank, local expert): ``rows`` in all, an eighth of the experts 8 times as popular."""
    p = torch.ones(local, device="cuda")
    p[: max(1, local // 8)] = 8.0
    to = torch.multinomial(p.repeat(ep), rows, replacement=True, generator=gen)
    return torch.bincount(to, minlength=ep * local).view(ep, local).to(torch.int32)


def _local(case):
    m = MODELS[case["model"]]
    return m["local"] if case["model"] == "qwen3-share" else m["E"] // case["ep"]


class _Group:
    """The process group's size and rank, all that the expert module asks of it."""

    def __init__(self, size):
        self.group_size, self.local_rank, self.in_participant = size, 0, True


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "layer":
        m = MODELS[case["model"]]
        mode = case["mode"]
        x = _normal(gen, (case["tokens"], m["H"]), 1.0, torch.float32 if mode == "fp32" else torch.bfloat16)
        logits = _logits(m, x, gen)
        w_gu, w_d, scales = _expert_weights(m, gen, mode, m["local"])
        kw = dict(renormalize=m["renorm"])
        if m["shared"]:
            kw.update(shared_gate_up=_normal(gen, (2 * m["shared"], m["H"]), 0.02),
                      shared_down=_normal(gen, (m["H"], m["shared"]), 0.02))
        if m["local"] < m["E"]:
            kw.update(expert_range=(0, m["local"]))
        if scales is not None:
            kw.update(w_scales=scales, w8a8=mode == "w8a8")
        if mode == "precise":
            kw.update(h_split=True)
        if case["gate"] == "sigmoid":
            kw.update(scoring_func="sigmoid", n_group=8, topk_group=4, renormalize=True, routed_scaling_factor=2.5,
                      e_score_correction_bias=_normal(gen, (m["E"],), 0.1, torch.float32))
        return dict(kind=kind, x=x, logits=logits, k=m["k"], w_gu=w_gu, w_d=w_d, kw=kw)
    if kind == "experts":
        m = MODELS[case["model"]]
        ep, local = case["ep"], _local(case)
        w_gu, w_d, scales = _expert_weights(m, gen, case["mode"], local)
        with torch.device("meta"):   # the module's own empty parameters are replaced at once
            mod = HipFusedMoE(0, m["H"], m["I"], "silu", False, False, local * ep, _Group(ep), _Group(1),
                              torch.arange(local * ep).view(ep, local))
        mod.experts_gate_up_weight = torch.nn.Parameter(w_gu, requires_grad=False)
        mod.experts_down_weight = torch.nn.Parameter(w_d, requires_grad=False)
        mod.w_scales = scales
        return dict(kind=kind, mod=mod, x=_normal(gen, (case["rows"], m["H"])), counts=_counts(case["rows"], ep, local, gen))
    if kind == "front":
        f = FRONTS[case["model"]]
        T = case["tokens"]
        st = dict(kind=kind, f=f, hidden=_normal(gen, (T, f["H"])), residual=_normal(gen, (T, f["H"])),
                  norm_w=(1.0 + _normal(gen, (f["H"],), 0.1, torch.float32)).to(torch.bfloat16),
                  gate_w=_normal(gen, (f["E"], f["H"]), 0.02))
        if f["grouped"]:
            st["bias"] = _normal(gen, (f["E"],), 0.1, torch.float32)
        return st
    m = MODELS[case["model"]]
    local = m["local"]
    blocks = _counts(case["rows"], case["ep"], local, gen)
    experts = [_normal(gen, (2 * m["I"], m["H"]), 0.02) for _ in range(local)]
    return dict(kind=kind, a=_normal(gen, (case["rows"], m["H"])), experts=experts * case["ep"],
                blocks=[int(b) for b in blocks.reshape(-1).tolist()])


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return fused_moe(state["x"], state["logits"], state["k"], state["w_gu"], state["w_d"], **state["kw"])
    if kind == "experts":
        return state["mod"].forward_ep(state["x"], state["counts"])
    if kind == "front":
        f = state["f"]
        res, normed, logits = ops.moe_prologue(state["hidden"], state["residual"], state["norm_w"], EPS, state["gate_w"],
                                               logits_bf16=not f["grouped"])
        if f["grouped"]:
            ids, w = ops.router_grouped_topk(logits, f["k"], 8, 4, state["bias"], True, 2.5)
        else:
            ids, w = ops.router_topk(logits, f["k"])
        return dict(residual=res, normed=normed, logits=logits, ids=ids, weights=w)
    return torch.ops.ops.hip_grouped_gemm_single(state["a"], state["experts"], state["blocks"])


# ------------------------------------------------------------------------------------------------ work
def work(case):
    kind = case["kind"]
    if kind == "front":
        f, T = FRONTS[case["model"]], case["tokens"]
        return dict(bytes=4.0 * T * f["H"] * 2 + f["H"] * 2 + f["E"] * f["H"] * 2 + T * f["E"] * 4 + T * f["k"] * 8,
                    flops=2.0 * T * f["H"] * f["E"])
    m = MODELS[case["model"]]
    H, I = m["H"], m["I"]
    if kind == "gemm":
        n = case["rows"]
        touched = _touched(_hot_shares(m["local"]), n)
        return dict(bytes=touched * 2.0 * I * H * 2 + n * (H + 2.0 * I) * 2, flops=4.0 * n * H * I)
    wb = {"bf16": 2, "precise": 2, "fp32": 4, "w8a8": 1, "w8a16": 1}[case["mode"]]
    if kind == "experts":
        n, local = case["rows"], _local(case)
        touched = _touched(_hot_shares(local), n)
        return dict(bytes=touched * (3.0 * H * I * wb + (2 * I + H) * 4 * (wb == 1)) + 2.0 * n * H * 2, flops=6.0 * n * H * I)
    T, E, k, local = case["tokens"], m["E"], m["k"], m["local"]
    xb = 4 if case["mode"] == "fp32" else 2
    if m["routing"] == "hotcold":
        n = T * k / 4.0
        touched = _touched(_hot_shares(local), n)
    else:
        n = T * k
        p = [r ** -1.2 for r in range(1, E + 1)] if m["routing"] == "zipf" else [1.0] * E
        touched = _touched([v / sum(p) for v in p], n)
    return dict(bytes=touched * (3.0 * H * I * wb + (2 * I + H) * 4 * (wb == 1)) + 3.0 * H * m["shared"] * 2
                + 2.0 * T * H * xb + T * E * 4.0,
                flops=6.0 * n * H * I + 6.0 * T * H * m["shared"])


def _hot_shares(local):
    p = [8.0 if e < max(1, local // 8) else 1.0 for e in range(local)]
    return [v / sum(p) for v in p]


def _touched(p, n):
    """Experts with at least one of n independent rows, on average (at least one)."""
    return max(1.0, sum(1.0 - (1.0 - v) ** n for v in p))


# ------------------------------------------------------------------------------------------------ exactness
def tolerance(case):
    """About four times the error against ``exact`` of this path as first measured, which is what the
    data types give: one bf16 rounding of h and one of the output (1.7e-3 each for N(0, 1) values), fp32
    sums over up to 14336 terms, e4m3 codes of h that flip with its last bf16 bit."""
    if case["kind"] == "front":
        # residual and normed differ by bf16 roundings that flip; ids by near-ties of the logits
        return dict(rel=1e-2, max=0.5, differ=5e-3)
    if case["kind"] == "layer":
        if case["mode"] == "fp32":
            return dict(rel=5e-6, max=5e-5)
    return dict(rel=1e-2, max=5e-2)


def _silu(g):
    return g / (1.0 + torch.exp(-g))


def _expert(x, w_gu, w_d, s_gu=None, s_d=None, w8a8=False):
    """One expert's MLP on rows x in 64 bits; with w8a8 the rows and h quantised as the mode says."""
    I = w_d.shape[1]
    scale = 1.0
    if w8a8:
        q, s = _rows_to_fp8(x)
        x, scale = q, s.double()[:, None]
    gu = (x.double() @ w_gu.double().T) * scale
    if s_gu is not None:
        gu = gu * s_gu.double()
    h = _silu(gu[:, :I]) * gu[:, I:]
    scale = 1.0
    if w8a8:
        q, s = _rows_to_fp8(h.to(torch.bfloat16))
        h, scale = q.double(), s.double()[:, None]
    y = (h @ w_d.double().T) * scale
    return y if s_d is None else y * s_d.double()


def _sigmoid_gate(logits, bias, k):
    T, E = logits.shape
    score = torch.sigmoid(logits.double())
    choice = score + bias.double()
    by_group = choice.view(T, 8, E // 8)
    kept = by_group.topk(2, dim=-1).values.sum(-1).topk(4, dim=-1).indices
    mask = torch.zeros(T, 8, device=logits.device, dtype=torch.bool).scatter_(1, kept, True)
    choice = torch.where(mask[:, :, None], by_group, torch.zeros_like(by_group)).view(T, E)
    ids = torch.sort(choice, dim=-1, descending=True, stable=True).indices[:, :k]
    w = score.gather(1, ids)
    return ids, w / (w.sum(-1, keepdim=True) + 1e-20) * 2.5


def _softmax_gate(logits, k, renorm):
    p = torch.softmax(logits.double(), dim=-1)
    ids = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :k]   # ties to the lower id
    w = p.gather(1, ids)
    return ids, w / w.sum(-1, keepdim=True) if renorm else w


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "layer":
        kw, x = st["kw"], st["x"]
        if case["gate"] == "sigmoid":
            ids, w = _sigmoid_gate(st["logits"], kw["e_score_correction_bias"], st["k"])
        else:
            ids, w = _softmax_gate(st["logits"], st["k"], kw["renormalize"])
        out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
        scales = kw.get("w_scales")
        for e in range(st["w_gu"].shape[0]):
            tok, slot = torch.nonzero(ids == e, as_tuple=True)
            if tok.numel() == 0:
                continue
            y = _expert(x[tok], st["w_gu"][e], st["w_d"][e], None if scales is None else scales[0][e],
                        None if scales is None else scales[1][e], kw.get("w8a8", False))
            out.index_add_(0, tok, y * w[tok, slot][:, None])
        if "shared_gate_up" in kw:
            out += _expert(x, kw["shared_gate_up"], kw["shared_down"])
        return out
    if kind == "experts":
        mod, x = st["mod"], st["x"]
        out = torch.empty(x.shape, dtype=torch.float64, device="cuda")
        at, local = 0, mod.num_physical_experts
        for s, n in enumerate(st["counts"].reshape(-1).tolist()):
            if n:
                e = s % local
                sc = (None, None) if mod.w_scales is None else (mod.w_scales[0][e], mod.w_scales[1][e])
                out[at:at + n] = _expert(x[at:at + n], mod.experts_gate_up_weight[e], mod.experts_down_weight[e], *sc)
            at += n
        return out
    if kind == "front":
        f = st["f"]
        res = (st["residual"].double() + st["hidden"].double()).to(torch.bfloat16).double()
        t = (res / torch.sqrt((res * res).mean(-1, keepdim=True) + EPS)).to(torch.bfloat16).double()
        normed = (st["norm_w"].double() * t).to(torch.bfloat16).double()
        logits = normed @ st["gate_w"].double().T
        if f["grouped"]:
            _, w = _sigmoid_gate(logits, st["bias"], f["k"])
        else:
            logits = logits.to(torch.bfloat16).double()
            _, w = _softmax_gate(logits, f["k"], True)
        return dict(residual=res, normed=normed, logits=logits, ids=None, weights=w)
    out, at = [], 0
    for n, b in zip(st["blocks"], st["experts"]):
        out.append(st["a"][at:at + n].double() @ b.double().T)
        at += n
    return torch.cat(out)
