"""Timed cases of the MoE expert path: what a program that trains or serves Qwen3-MoE layers calls.

A case is one pass through a public entry point on inputs that the program
already holds on the GPU:

  infer     SparseMoeBlock under no_grad: decode steps and prefill
  train     ops.moe_block forward and backward (with the aux loss), one or
            several microbatches per optimizer step, bf16 or fp32 modules
  ep_share  ops.experts forward and backward on an expert-parallel rank's
            receive buffer, Zipf-skewed routing, some local experts empty
  norm      norm_router_aux forward and backward: the decoder layer's norm,
            router and aux loss before the experts
  dispatch  TokenDispatcher dispatch and combine, forward and backward

`listed()` holds the fixed cases, `draw()` draws others of the same ranges.
`exact()` restates each case in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch

from parallel_amd import ExpertPartition, MoeConfig, SparseMoeBlock, TokenDispatcher, norm_router_aux, ops

AUX_COEF = 0.001
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
# (hidden, experts, top_k, intermediate): the benchmark's two layers, the fp32
# layer of its CPU configuration, and two generic smaller ones.
LAYER_30B = dict(hidden=2048, experts=128, top_k=8, inter=768)
LAYER_235B = dict(hidden=4096, experts=128, top_k=8, inter=1536)
LAYER_TINY = dict(hidden=256, experts=8, top_k=2, inter=128)
LAYER_SMALL = dict(hidden=1024, experts=32, top_k=4, inter=512)
LAYER_MID = dict(hidden=1536, experts=64, top_k=6, inter=640)


def listed() -> list[dict]:
    return [
        # one sequence decoding: a single token through the layer, latency and launches
        dict(name="decode_1", kind="infer", tokens=1, dtype="bf16", **LAYER_30B),
        # a serving batch decoding: most experts hit by a few rows each, the weights stream once
        dict(name="decode_48", kind="infer", tokens=48, dtype="bf16", **LAYER_30B),
        # prefill of one prompt of an odd length
        dict(name="prefill_1531", kind="infer", tokens=1531, dtype="bf16", **LAYER_30B),
        # a short training sequence under bf16 autocast (bf16 router logits)
        dict(name="train_301_amp", kind="train", tokens=301, micro=1, dtype="bf16", bf16_logits=True, skew=0.0,
             **LAYER_30B),
        # the benchmark's headline step: 4096 tokens of the 30B layer
        dict(name="train_4096", kind="train", tokens=4096, micro=1, dtype="bf16", bf16_logits=False, skew=0.0,
             **LAYER_30B),
        # gradient accumulation over two microbatches (16384 tokens), imbalanced router
        dict(name="train_2x8192_accum", kind="train", tokens=8192, micro=2, dtype="bf16", bf16_logits=False, skew=0.5,
             **LAYER_30B),
        # the 235B layer at 8192 tokens
        dict(name="train_8192_235b", kind="train", tokens=8192, micro=1, dtype="bf16", bf16_logits=False, skew=0.0,
             **LAYER_235B),
        # expert-parallel rank of two: 64 local experts, rows of 2 x 4096 tokens, Zipf(1.2) routing
        dict(name="ep_share_zipf", kind="ep_share", tokens=4096, sources=2, local=64, alpha=1.2, dtype="bf16",
             **LAYER_30B),
        # the fp32 modules' tiny block (the CPU-runnable configuration)
        dict(name="train_512_fp32", kind="train", tokens=512, micro=1, dtype="fp32", bf16_logits=False, skew=0.0,
             **LAYER_TINY),
        # a small fp32 layer in training (full-precision runs and ablations)
        dict(name="train_2048_fp32", kind="train", tokens=2048, micro=1, dtype="fp32", bf16_logits=False, skew=0.0,
             **LAYER_SMALL),
        # the step before the experts in a masked (padded) training batch
        dict(name="norm_router_5000", kind="norm", tokens=5000, dtype="bf16", **LAYER_30B),
        # sequence-parallel dispatch to expert owners and back
        dict(name="dispatch_4096", kind="dispatch", tokens=4096, ep=2, dtype="bf16", **LAYER_30B),
    ]


def _tokens(rng, lo: int, hi: int) -> int:
    """Log-uniform token count; odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["infer", "infer", "infer", "train", "train", "train", "train", "fp32", "fp32", "ep_share",
                       "norm", "dispatch"])
    layer = dict(rng.choice([LAYER_30B, LAYER_30B, LAYER_30B, LAYER_MID, LAYER_SMALL]))
    if kind == "infer":
        if rng.random() < 0.15:
            layer = dict(LAYER_235B)
        return dict(kind="infer", tokens=_tokens(rng, 1, 4096), dtype="bf16", **layer)
    if kind == "train":
        hi = 12000
        if rng.random() < 0.15:
            layer, hi = dict(LAYER_235B), 4096
        micro = rng.choice([1, 1, 2])
        return dict(kind="train", tokens=_tokens(rng, 64, hi // micro), micro=micro, dtype="bf16",
                    bf16_logits=rng.random() < 0.4, skew=rng.choice([0.0, 0.0, 0.25, 0.5]), **layer)
    if kind == "fp32":
        layer = dict(rng.choice([LAYER_TINY, LAYER_SMALL]))
        return dict(kind="train", tokens=_tokens(rng, 64, 2048), micro=1, dtype="fp32", bf16_logits=False,
                    skew=rng.choice([0.0, 0.5]), **layer)
    if kind == "ep_share":
        layer = dict(rng.choice([LAYER_30B, LAYER_MID]))
        sources = rng.choice([2, 4])
        return dict(kind="ep_share", tokens=_tokens(rng, 128, 8192 // sources), sources=sources,
                    local=layer["experts"] // sources, alpha=round(rng.uniform(0.6, 1.3), 2), dtype="bf16", **layer)
    if kind == "norm":
        return dict(kind="norm", tokens=_tokens(rng, 64, 16384), dtype="bf16", **layer)
    return dict(kind="dispatch", tokens=_tokens(rng, 64, 8192), ep=rng.choice([1, 2, 2] if layer["top_k"] % 4 else
                                                                              [1, 2, 4]), dtype="bf16", **layer)


# ------------------------------------------------------------------- inputs


class _Rand:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.gen, device="cuda", dtype=dtype).mul_(std)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device="cuda", dtype=torch.float64)


def _weights(case, r: _Rand, experts: int):
    dt = DTYPES[case["dtype"]]
    H, I = case["hidden"], case["inter"]
    return r.normal(experts, 2 * I, H, std=0.02, dtype=dt), r.normal(experts, H, I, std=0.02, dtype=dt)


def _receive_count(case) -> int:
    """Rows of the receive buffer: the rank's share of a uniform draw."""
    return case["sources"] * case["tokens"] * case["top_k"] * case["local"] // case["experts"]


def _receive_rows(case, r: _Rand):
    """(row expert ids [R], row scores [R]) of rank 0's receive buffer: source-rank-major, flat (token, k)
    order within a source; top-k distinct experts with weight rank^-alpha, four local experts empty.
    The buffer holds the first R rows (further tokens of the sources fill it where the draw gave fewer)."""
    E, k, local, R = case["experts"], case["top_k"], case["local"], _receive_count(case)
    order = torch.argsort(r.uniform(E))
    logw = torch.empty(E, dtype=torch.float64, device="cuda")
    logw[order] = -case["alpha"] * torch.log(torch.arange(1, E + 1, dtype=torch.float64, device="cuda"))
    logw[torch.argsort(r.uniform(local))[:4]] = -math.inf
    ids, scores, have = [], [], 0
    while have < R:
        u = r.uniform(case["sources"] * case["tokens"], E).clamp_(1e-12, 1 - 1e-12)
        i = torch.topk(logw - torch.log(-torch.log(u)), k, dim=1).indices
        s = torch.softmax(r.normal(*i.shape), dim=1)
        mine = i < local
        ids.append(i[mine])
        scores.append(s[mine])
        have += ids[-1].numel()
    return torch.cat(ids)[:R].contiguous(), torch.cat(scores)[:R].contiguous()


def _owner_ids(case, r: _Rand):
    """[T, k] distinct expert ids, k / ep of every owner rank's experts in a random slot order."""
    T, E, k, ep = case["tokens"], case["experts"], case["top_k"], case["ep"]
    local = E // ep
    ids = [torch.argsort(r.uniform(T, local), dim=1)[:, :k // ep] + o * local for o in range(ep)]
    ids = torch.cat(ids, dim=1)
    return ids.gather(1, torch.argsort(r.uniform(T, k), dim=1)).contiguous()


def prepare(case: dict, seed: int) -> dict:
    r = _Rand(seed)
    dt = DTYPES[case["dtype"]]
    kind, T, H, E, k = case["kind"], case["tokens"], case["hidden"], case["experts"], case["top_k"]
    if kind == "infer":
        with torch.device("meta"):
            block = SparseMoeBlock(MoeConfig(H, E, k, case["inter"], norm_topk_prob=True)).eval()
        gu, dn = _weights(case, r, E)
        block.experts.gate_up_proj = torch.nn.Parameter(gu, requires_grad=False)
        block.experts.down_proj = torch.nn.Parameter(dn, requires_grad=False)
        block.gate.weight = torch.nn.Parameter(r.normal(E, H, std=0.02, dtype=dt), requires_grad=False)
        return dict(case=case, block=block, x=r.normal(1, T, H, dtype=dt))
    if kind == "train":
        gu, dn = _weights(case, r, E)
        rw = r.normal(E, H, std=(1.0 / math.sqrt(H)) if case["skew"] else 0.02, dtype=dt)
        bias = r.normal(E, std=case["skew"]) if case["skew"] else None
        xs = [r.normal(T, H, dtype=dt).requires_grad_() for _ in range(case["micro"])]
        d_outs = [r.normal(T, H, dtype=dt) for _ in range(case["micro"])]
        return dict(case=case, gu=gu.requires_grad_(), dn=dn.requires_grad_(), rw=rw.requires_grad_(), bias=bias,
                    xs=xs, d_outs=d_outs, d_aux=torch.tensor(AUX_COEF, device="cuda"))
    if kind == "ep_share":
        ids, scores = _receive_rows(case, r)
        gu, dn = _weights(case, r, case["local"])
        return dict(case=case, rows=r.normal(ids.numel(), H, dtype=dt).requires_grad_(), ids=ids.unsqueeze(1),
                    scores=scores.unsqueeze(1).requires_grad_(), gu=gu.requires_grad_(), dn=dn.requires_grad_(),
                    d_out=r.normal(ids.numel(), H, dtype=dt))
    if kind == "norm":
        mask = torch.ones(1, T, device="cuda")
        mask[:, T - T // 8:] = 0.0  # the last eighth is padding
        return dict(case=case, hidden=r.normal(1, T, H, std=1.5, dtype=dt).requires_grad_(),
                    gamma=(1.0 + r.normal(H, std=0.1)).to(dt).requires_grad_(),
                    rw=r.normal(E, H, std=0.02, dtype=dt).requires_grad_(), mask=mask, d_x=r.normal(1, T, H, dtype=dt),
                    d_scores=r.normal(T, k), d_aux=torch.tensor(AUX_COEF, device="cuda"))
    dispatcher = TokenDispatcher(ExpertPartition(E, case["ep"], 0), None)
    ids = _owner_ids(case, r)
    return dict(case=case, dispatcher=dispatcher, hidden=r.normal(T, H, dtype=dt).requires_grad_(), ids=ids,
                scores=torch.softmax(r.normal(T, k), dim=1), d_out=r.normal(T, H, dtype=dt))


# --------------------------------------------------------------------- pass


def run(state: dict):
    case = state["case"]
    kind, k = case["kind"], case["top_k"]
    if kind == "infer":
        with torch.no_grad():
            return state["block"](state["x"])
    if kind == "train":
        params = (state["rw"], state["gu"], state["dn"])
        for p in params:
            p.grad = None
        results = []
        for x, d_out in zip(state["xs"], state["d_outs"]):
            x.grad = None
            out, logits, _scores, _idx, aux = ops.moe_block(x, *params, k, True, None, state["bias"],
                                                            accumulate_grad=case["micro"] > 1,
                                                            bf16_logits=case["bf16_logits"])
            torch.autograd.backward([out, aux], [d_out, state["d_aux"]])
            results.append((out.detach(), logits.detach(), aux.detach(), x.grad))
        return results, [p.grad for p in params]
    if kind == "ep_share":
        leaves = (state["rows"], state["scores"], state["gu"], state["dn"])
        for p in leaves:
            p.grad = None
        out = ops.experts(state["rows"], state["ids"], state["scores"], state["gu"], state["dn"])
        out.backward(state["d_out"])
        return out.detach(), [p.grad for p in leaves]
    if kind == "norm":
        leaves = (state["hidden"], state["gamma"], state["rw"])
        for p in leaves:
            p.grad = None
        x, (logits, scores, idx), aux = norm_router_aux(*leaves, k, attention_mask=state["mask"])
        torch.autograd.backward([x, scores, aux], [state["d_x"], state["d_scores"], state["d_aux"]])
        return x.detach(), logits.detach(), scores.detach(), idx, aux.detach(), [p.grad for p in leaves]
    hidden = state["hidden"]
    hidden.grad = None
    received, experts, scores, sent = state["dispatcher"].dispatch(hidden, state["ids"], state["scores"])
    out = state["dispatcher"].combine(received, sent)
    out.backward(state["d_out"])
    return received.detach(), experts, scores, out.detach(), hidden.grad


# ------------------------------------------------------- work and tolerances


def _expected_experts(T: int, k: int, E: int) -> float:
    """Experts that at least one of T tokens picks, k of E at random each."""
    return E * (1.0 - (1.0 - k / E) ** T)


def work(case: dict) -> dict:
    kind, T, H, E, k, I = (case[n] for n in ("kind", "tokens", "hidden", "experts", "top_k", "inter"))
    b = 4 if case["dtype"] == "fp32" else 2
    expert = 3 * I * H * b  # one expert's weights
    if kind == "infer":
        return {"bytes": _expected_experts(T, k, E) * expert + E * H * b + 2 * T * H * b,
                "flops": T * k * 6.0 * H * I + 2.0 * T * E * H}
    if kind == "train":
        # x, d_out in, out, dx out; the weights read once, their gradients written once
        n = case["micro"] * T
        return {"bytes": 4 * n * H * b + 4 * n * E + 2 * (E * expert + E * H * b),
                "flops": n * (k * 18.0 * H * I + 6.0 * E * H)}
    if kind == "ep_share":
        rows = _receive_count(case)
        return {"bytes": 4 * rows * H * b + 2 * case["local"] * expert, "flops": rows * 18.0 * H * I}
    if kind == "norm":
        return {"bytes": 4 * T * H * b + 2 * E * H * b + T * (4 * E + 16 * k), "flops": 6.0 * T * E * H}
    share = T * k / case["ep"]
    return {"bytes": T * H * b + share * (H * b + 12) + T * H * b + 2 * T * H * b + T * k * 12, "flops": 0}


def tolerance(case: dict):
    if case["dtype"] == "fp32":
        # measured against float64: 3e-7 to 1.1e-6 (sums of up to 2048 terms), times four and as much again
        # for the products' own order
        return {"rel": 1e-5}
    # measured against float64: 2e-3 to 5e-3 of bf16 results through bf16 intermediates, times about four for the
    # largest; two router logits of nearly the same value may select the experts in the other order
    return {"rel": 1.5e-2, "differ": 1e-3}


# -------------------------------------------------------------- float64 oracle


def _route(logits, k):
    """(probabilities, renormalised scores, indices) of the top k, ties to the lower index."""
    p = torch.softmax(logits, dim=1)
    idx = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :k]
    top = p.gather(1, idx)
    return p, top / top.sum(1, keepdim=True), idx


def _experts64(x, ids, scores, gu, dn, d_out=None):
    """The expert layer on float64 rows, and with d_out its gradients (dx, d_scores, d_gu, d_dn)."""
    T, H = x.shape
    k = ids.shape[1]
    E, I = gu.shape[0], gu.shape[1] // 2
    flat = ids.reshape(-1)
    out = torch.zeros_like(x)
    grads = None
    if d_out is not None:
        grads = [torch.zeros_like(x), torch.zeros(T * k, dtype=torch.float64, device=x.device),
                 torch.zeros(gu.shape, dtype=torch.float64, device=x.device),
                 torch.zeros(dn.shape, dtype=torch.float64, device=x.device)]
    for e in range(E):
        slots = torch.nonzero(flat == e).squeeze(1)
        if slots.numel() == 0:
            continue
        tok, s = slots // k, scores.reshape(-1)[slots].unsqueeze(1)
        w1, w2 = gu[e].double(), dn[e].double()
        rows = x[tok]
        pre = rows @ w1.t().contiguous()
        gate, up = pre[:, :I], pre[:, I:]
        sig = torch.sigmoid(gate)
        act = gate * sig * up
        y = act @ w2.t().contiguous()
        out.index_add_(0, tok, s * y)
        if grads is not None:
            g = d_out[tok]
            grads[1][slots] = (g * y).sum(1)
            dy = s * g
            d_act = dy @ w2
            d_pre = torch.cat([d_act * up * sig * (1 + gate * (1 - sig)), d_act * gate * sig], dim=1)
            grads[0].index_add_(0, tok, d_pre @ w1)
            grads[2][e] = d_pre.t().contiguous() @ rows
            grads[3][e] = dy.t().contiguous() @ act
    if grads is not None:
        grads[1] = grads[1].view(T, k)
    return out, grads


def _router_grad(logits, k, idx, d_scores, weight, d_aux):
    """d_logits of the renormalised top-k scores and of the Switch aux loss (token weights `weight`); and the loss."""
    E = logits.shape[1]
    z = logits.detach().requires_grad_()
    p = torch.softmax(z, dim=1)
    top = p.gather(1, idx)
    scores = top / top.sum(1, keepdim=True)
    counts = torch.zeros_like(p).scatter_(1, idx, 1.0)
    total = weight.sum()
    aux = E * ((counts * weight.unsqueeze(1)).sum(0) / total * ((p * weight.unsqueeze(1)).sum(0) / total)).sum()
    (dz,) = torch.autograd.grad([scores, aux], [z], [d_scores, torch.tensor(d_aux, dtype=torch.float64, device=z.device)])
    return dz, aux.detach()


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    kind, k = case["kind"], case["top_k"]
    with torch.no_grad():
        if kind == "infer":
            block, x = st["block"], st["x"][0].double()
            _, scores, idx = _route(x @ block.gate.weight.double().t().contiguous(), k)
            return _experts64(x, idx, scores, block.experts.gate_up_proj, block.experts.down_proj)[0].unsqueeze(0)
        if kind == "train":
            rw = st["rw"].double()
            results, grads = [], None
            for x, d_out in zip(st["xs"], st["d_outs"]):
                x = x.detach().double()
                logits = x @ rw.t().contiguous()
                if st["bias"] is not None:
                    logits = logits + st["bias"].double()
                if case["bf16_logits"]:
                    logits = logits.to(torch.bfloat16).double()  # the logits tensor itself is bf16
                _, scores, idx = _route(logits, k)
                if case["bf16_logits"]:
                    scores = scores.to(torch.bfloat16).double()
                out, (dx, d_scores, d_gu, d_dn) = _experts64(x, idx, scores, st["gu"], st["dn"], d_out.double())
                with torch.enable_grad():
                    dz, aux = _router_grad(logits, k, idx, d_scores,
                                           torch.ones(x.shape[0], dtype=torch.float64, device="cuda"), AUX_COEF)
                results.append((out, logits, aux, dx + dz @ rw))
                new = [dz.t().contiguous() @ x, d_gu, d_dn]
                grads = new if grads is None else [a.add_(b) for a, b in zip(grads, new)]
            return results, grads
        if kind == "ep_share":
            out, grads = _experts64(st["rows"].detach().double(), st["ids"], st["scores"].double(), st["gu"], st["dn"],
                                    st["d_out"].double())
            return out, grads
        if kind == "norm":
            h, gamma, rw = st["hidden"].detach()[0].double(), st["gamma"].double(), st["rw"].double()
            r = torch.rsqrt((h * h).mean(1, keepdim=True) + 1e-6)
            hs = h * r
            x = (hs.to(torch.bfloat16).double() * gamma).to(torch.bfloat16).double()  # the router reads the bf16 x
            logits = x @ rw.t().contiguous()
            _, scores, idx = _route(logits, k)
            with torch.enable_grad():
                dz, aux = _router_grad(logits, k, idx, st["d_scores"].double(), st["mask"].reshape(-1).double(),
                                       AUX_COEF)
            g = st["d_x"][0].double() + dz @ rw
            dhs = g * gamma
            dh = r * dhs - r ** 3 * h * (dhs * h).mean(1, keepdim=True)
            return (hs * gamma).unsqueeze(0), logits, scores, None, aux, [dh.unsqueeze(0), (g * hs).sum(0),
                                                                           dz.t().contiguous() @ x]
        owner = st["ids"] // (case["experts"] // case["ep"])
        mine = (owner == 0)
        count = mine.sum(1, keepdim=True).double()
        rows = torch.nonzero(mine.reshape(-1)).squeeze(1)
        hidden = st["hidden"].detach().double()
        return (hidden[rows // k], None, st["scores"].double().reshape(-1)[rows].unsqueeze(1), count * hidden,
                count * st["d_out"].double())
