"""The routing chain and its operators as a serving program calls them, at the
sizes this library is used for.

A case is a dict of plain values. "path" says which public entry one pass goes
through:

  tokens    chain_from_tokens: router GEMM, top-2 gate, histogram + scan,
            permute, expert GEMM and weighted unpermute of one MoE layer;
  logits    chain_from_logits: the same layer behind a router of the caller's;
  routes    chain_from_route_ids: the layer behind a router and gate of the
            caller's, any top_k;
  histogram histogram_exclusive_scan over a batch of route ids;
  staged    histogram_exclusive_scan, token_permute, grouped_gemm and unpermute
            called one by one (a program that keeps the permuted rows, or puts
            its own work between the stages).

A pass is given device buffers, argument structs and a workspace that the
program keeps, and enqueues the call(s) on the current stream.
"""
from __future__ import annotations

import math

import torch

import raggedroute_amd as rr

DEVICE = "cuda:0"


def listed() -> list[dict]:
    return [
        # A decode step's handful of tokens: launches and latency are all there is.
        dict(name="tokens_decode", path="tokens", tokens=64, experts=16, hidden=64, output=64, skew=0.0),
        # A short prefill at the shape the chain's published numbers are quoted on.
        dict(name="tokens_short", path="tokens", tokens=512, experts=64, hidden=128, output=128, skew=0.0),
        # The headline batch: 4096 tokens over 64 narrow experts.
        dict(name="tokens_headline", path="tokens", tokens=4096, experts=64, hidden=256, output=128, skew=0.0),
        # A batch that nothing was rounded for: odd tokens, widths off every vector size.
        dict(name="tokens_ragged", path="tokens", tokens=1777, experts=40, hidden=333, output=95, skew=0.0),
        # A mid-size layer: more rows than a decode, wider than the narrow experts.
        dict(name="tokens_mid", path="tokens", tokens=2048, experts=64, hidden=1024, output=512, skew=0.0),
        # Large-batch prefill of a fine-grained MoE layer with log-Zipf skewed routing.
        dict(name="tokens_prefill", path="tokens", tokens=16384, experts=128, hidden=2048, output=768, skew=1.0),
        # The headline batch behind the caller's own router: skewed logits, some exact ties.
        dict(name="logits_skewed", path="logits", tokens=4096, experts=64, hidden=256, output=128, skew=1.1),
        # The caller's own gate with four routes a token, skewed ids, permuted rows kept.
        dict(name="routes_top4", path="routes", tokens=2048, experts=64, hidden=128, output=128, top_k=4,
             skew=1.4, keep_rows=True),
        # Eight routes a token at the largest route count of the post-route chain's configurations.
        dict(name="routes_top8", path="routes", tokens=8192, experts=64, hidden=64, output=64, top_k=8,
             skew=0.0, keep_rows=False),
        # Load statistics over a million routes, half of them on one hot expert.
        dict(name="histogram_hot", path="histogram", routes=1 << 20, experts=256, hot=0.5),
        # The operators one by one on a ragged problem: odd tokens and widths, an expert without tokens.
        dict(name="staged_ragged", path="staged", tokens=3001, experts=9, active=8, hidden=1023, output=1535, skew=0.6),
        # The operators one by one at Mixtral's layer size, seven of eight experts active.
        dict(name="staged_wide", path="staged", tokens=8192, experts=8, active=7, hidden=4096, output=14336, skew=1.2),
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo: int, hi: int, odd: bool) -> int:
    """A row width: any number, or (most models) a multiple of 32."""
    n = _log_uniform(rng, lo, hi)
    return n if odd else max(lo, n // 32 * 32)


def draw(rng) -> dict:
    path = rng.choice(["tokens", "tokens", "tokens", "logits", "routes", "histogram", "staged", "staged"])
    odd = rng.random() < 0.4
    if path == "histogram":
        return dict(path=path, routes=_log_uniform(rng, 8192, 1 << 20), experts=_log_uniform(rng, 8, 256),
                    hot=rng.choice([0.0, 0.5]))
    if path == "routes":
        top_k = rng.choice([2, 4, 8])
        return dict(path=path, tokens=_log_uniform(rng, 64, 8192), experts=_log_uniform(rng, 16, 128),
                    hidden=_width(rng, 64, 256, odd), output=_width(rng, 64, 256, odd), top_k=top_k,
                    skew=rng.choice([0.0, 1.4]), keep_rows=rng.random() < 0.5)
    if path == "staged":
        experts = _log_uniform(rng, 4, 64)
        return dict(path=path, tokens=_log_uniform(rng, 512, 8192), experts=experts,
                    active=max(2, experts - rng.randrange(2)), hidden=_width(rng, 256, 4096, odd),
                    output=_width(rng, 512, 8192, odd), skew=rng.choice([0.0, 0.6, 1.2]))
    return dict(path=path, tokens=_log_uniform(rng, 64, 16384), experts=_log_uniform(rng, 8, 128),
                hidden=_width(rng, 64, 2048, odd), output=_width(rng, 64, 768, odd),
                skew=rng.choice([0.0, 1.0]))


class _Inputs:
    """Seeded device tensors: every draw of one state comes from one generator."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std: float = 1.0) -> torch.Tensor:
        return torch.randn(*shape, device=DEVICE, generator=self.gen).mul_(std)

    def uniform(self, *shape) -> torch.Tensor:
        return torch.rand(*shape, device=DEVICE, generator=self.gen)

    def popularity(self, experts: int, skew: float) -> torch.Tensor:
        """log p(e) of a Zipf(skew) popularity dealt to the experts at random."""
        rank = torch.randperm(experts, device=DEVICE, generator=self.gen)
        return -skew * torch.log(rank.float() + 1.0)

    def distinct_ids(self, tokens: int, top_k: int, experts: int, skew: float) -> torch.Tensor:
        """top_k distinct experts a token, drawn without replacement by popularity."""
        gumbel = -torch.log(-torch.log(self.uniform(tokens, experts).clamp_(1e-7, 1.0 - 1e-6)))
        return torch.topk(gumbel + self.popularity(experts, skew), top_k, dim=1).indices.int().contiguous()


def _inputs(case: dict, seed: int) -> dict:
    g = _Inputs(seed)
    path = case["path"]
    e = case["experts"]
    if path == "histogram":
        r = case["routes"]
        ids = torch.randint(0, e, (r,), device=DEVICE, generator=g.gen, dtype=torch.int32)
        if case["hot"] > 0:
            hot = torch.randint(0, e, (1,), device=DEVICE, generator=g.gen, dtype=torch.int32)
            ids = torch.where(g.uniform(r) < case["hot"], hot, ids)
        return {"ids": ids.contiguous()}
    t, k, n = case["tokens"], case["hidden"], case["output"]
    sd = 1.0 / math.sqrt(k)
    out = {"x": g.normal(t, k), "expert_weights": g.normal(e, k, n, std=sd)}
    if path == "tokens":
        wr = g.normal(k, e, std=sd)
        if case["skew"] > 0:  # a router bias inside the GEMM: a constant feature and its row
            out["x"][:, k - 1] = 1.0
            wr[k - 1, :] = g.popularity(e, case["skew"])
        out["router_weights"] = wr
    elif path == "logits":
        logits = g.normal(t, e) + g.popularity(e, case["skew"])
        tie = g.uniform(t) < 0.02  # these rows' third choice equals their second
        order = torch.argsort(logits, dim=1, descending=True)
        second = logits.gather(1, order[:, 1:2])
        third = logits.gather(1, order[:, 2:3])
        logits.scatter_(1, order[:, 2:3], torch.where(tie[:, None], second, third))
        out["logits"] = logits
    else:
        top_k = case.get("top_k", 2)
        out["ids"] = g.distinct_ids(t, top_k, case.get("active", e), case["skew"])
        w = g.uniform(t, top_k) + 0.01
        out["weights"] = w / w.sum(dim=1, keepdim=True)
    return out


def prepare(case: dict, seed: int) -> dict:
    inp = _inputs(case, seed)
    stream = torch.cuda.current_stream().cuda_stream
    i32 = dict(dtype=torch.int32, device=DEVICE)
    f32 = dict(dtype=torch.float32, device=DEVICE)
    e = case["experts"]
    out = {"counts": torch.empty(e, **i32), "offsets": torch.empty(e + 1, **i32)}
    state = {"case": case, "inputs": inp, "outputs": out}
    p = {name: v.data_ptr() for name, v in out.items()}
    if case["path"] == "histogram":
        state["args"] = rr.HistogramExclusiveScanArgs(
            expert_ids=inp["ids"].data_ptr(), counts=p["counts"], offsets=p["offsets"],
            route_pairs=case["routes"], experts=e)
        state["context"] = rr.RuntimeContext(stream=stream)
        return state

    t, k, n, top_k = case["tokens"], case["hidden"], case["output"], case.get("top_k", 2)
    routes = t * top_k
    if case.get("keep_rows", True):
        out["x_permuted"] = torch.empty(routes, k, **f32)
    out["route_pos"] = torch.empty(routes, **i32)
    out["y_permuted"] = torch.empty(routes, n, **f32)
    out["y"] = torch.empty(t, n, **f32)
    if case["path"] in ("tokens", "logits"):
        if case["path"] == "tokens":
            out["logits"] = torch.empty(t, e, **f32)
        out["expert_ids"] = torch.empty(t, 2, **i32)
        out["route_weights"] = torch.empty(t, 2, **f32)
    p = {name: v.data_ptr() for name, v in {**inp, **out}.items()}

    def context(bytes_: int):
        ws = torch.empty(max(64, (bytes_ + 3) // 4), **i32)
        state.setdefault("workspaces", []).append(ws)
        return rr.RuntimeContext(stream=stream, workspace=ws.data_ptr(), workspace_bytes=ws.numel() * 4)

    if case["path"] in ("tokens", "logits"):
        state["args"] = rr.ChainArgs(
            x=p["x"], router_weights=p.get("router_weights"), logits=p["logits"], expert_ids=p["expert_ids"],
            route_weights=p["route_weights"], counts=p["counts"], offsets=p["offsets"],
            x_permuted=p["x_permuted"], route_pos=p["route_pos"], expert_weights=p["expert_weights"],
            y_permuted=p["y_permuted"], y=p["y"], tokens=t, experts=e, hidden=k, output=n)
        state["context"] = context(rr.get_chain_workspace_size(state["args"]))
    elif case["path"] == "routes":
        state["args"] = rr.RouteChainArgs(
            x=p["x"], expert_ids=p["ids"], route_weights=p["weights"], expert_weights=p["expert_weights"],
            counts=p["counts"], offsets=p["offsets"], x_permuted=p.get("x_permuted"),
            route_pos=p["route_pos"], y_permuted=p["y_permuted"], y=p["y"], tokens=t, experts=e,
            top_k=top_k, hidden=k, output=n)
        state["context"] = context(rr.get_route_chain_workspace_size(state["args"]))
    else:
        state["args"] = (
            rr.HistogramExclusiveScanArgs(expert_ids=p["ids"], counts=p["counts"], offsets=p["offsets"],
                                          route_pairs=routes, experts=e),
            rr.TokenPermuteArgs(x=rr.cview(p["x"]), expert_ids=p["ids"], offsets=p["offsets"],
                                x_permuted=rr.mview(p["x_permuted"]), route_pos=p["route_pos"],
                                tokens=t, experts=e, top_k=top_k, hidden=k),
            rr.GroupedGemmArgs(x_permuted=rr.cview(p["x_permuted"]),
                               expert_weights=rr.cview(p["expert_weights"]), offsets=p["offsets"],
                               y_permuted=rr.mview(p["y_permuted"]), experts=e, hidden=k, output=n,
                               max_expert_tokens=routes),
            rr.UnpermuteArgs(y_permuted=rr.cview(p["y_permuted"]), route_pos=p["route_pos"],
                             route_weights=rr.cview(p["weights"]), y=rr.mview(p["y"]), tokens=t,
                             top_k=top_k, output=n))
        state["context"] = context(rr.get_token_permute_workspace_size(state["args"][1]))
    return state


def _ok(status) -> None:
    if not status.ok():
        raise RuntimeError(status.message)


_ENTRY = {"tokens": rr.chain_from_tokens, "logits": rr.chain_from_logits, "routes": rr.chain_from_route_ids,
          "histogram": rr.histogram_exclusive_scan}


def run(state: dict) -> dict:
    context = state["context"]
    if state["case"]["path"] == "staged":
        histogram, permute, grouped, unpermute = state["args"]
        _ok(rr.histogram_exclusive_scan(histogram, context))
        _ok(rr.token_permute(permute, context))
        _ok(rr.grouped_gemm(grouped, context))
        _ok(rr.unpermute(unpermute, context))
    else:
        _ok(_ENTRY[state["case"]["path"]](state["args"], context))
    return state["outputs"]


def work(case: dict) -> dict:
    """Each input read once and each output written once (FP32 and int32), and the
    multiply-adds of the GEMMs and the combine. The expert weights count for the
    experts that are meant to be active."""
    e = case["experts"]
    if case["path"] == "histogram":
        return {"bytes": 4 * (case["routes"] + 2 * e + 1), "flops": 0}
    t, k, n, top_k = case["tokens"], case["hidden"], case["output"], case.get("top_k", 2)
    r = t * top_k
    floats = t * k + case.get("active", e) * k * n + r * n + t * n + r  # x, W, y_permuted, y, weights
    if case.get("keep_rows", True):
        floats += r * k
    ints = 2 * r + 2 * e + 1  # ids, route_pos, counts, offsets
    flops = 2 * r * k * n + 2 * r * n
    if case["path"] == "tokens":
        floats += k * e + t * e
        flops += 2 * t * k * e
    elif case["path"] == "logits":
        floats += t * e
    return {"bytes": 4 * (floats + ints), "flops": flops}


def tolerance(case: dict):
    """FP32 sums of K products. Against the float64 results below, the worst
    output is off by 2e-7 (K = 64), 4.6e-7 (K = 256), 9.1e-7 (K = 1024) and
    1.1e-6 (K = 4096) of its 2-norm; another order of the sums may show about
    four times that. Row maps, counts and ids are exact."""
    if case["path"] == "histogram":
        return "exact"
    return {"rel": 8e-7 + 9e-8 * math.sqrt(case["hidden"])}


def exact(case: dict, seed: int):
    """The same layer in float64 (routing decided on the float64 logits, ties to the lower expert)."""
    if case["path"] == "histogram":
        return None
    inp = _inputs(case, seed)
    t, e, n, top_k = case["tokens"], case["experts"], case["output"], case.get("top_k", 2)
    out = {"counts": None, "offsets": None, "route_pos": None}
    if case["path"] in ("tokens", "logits"):
        if case["path"] == "tokens":
            logits = inp["x"].double() @ inp["router_weights"].double()
            out["logits"] = logits
        else:
            logits = inp["logits"].double()
        order = torch.sort(logits, dim=1, descending=True, stable=True)
        ids = order.indices[:, :2]
        weights = torch.softmax(order.values[:, :2], dim=1)
        out["expert_ids"], out["route_weights"] = None, weights
    else:
        ids, weights = inp["ids"].long(), inp["weights"].double()
    flat = ids.reshape(-1)
    sorted_route = torch.sort(flat, stable=True).indices  # routes in segment order
    counts = torch.bincount(flat, minlength=e).tolist()
    x_permuted = inp["x"][sorted_route // top_k]
    if case.get("keep_rows", True):
        out["x_permuted"] = x_permuted.double()
    y_permuted = torch.zeros(t * top_k, n, dtype=torch.float64, device=DEVICE)
    row = 0
    for expert, rows in enumerate(counts):
        if rows:
            y_permuted[row:row + rows] = x_permuted[row:row + rows].double() @ inp["expert_weights"][expert].double()
            row += rows
    out["y_permuted"] = y_permuted
    position = torch.empty_like(sorted_route)
    position[sorted_route] = torch.arange(t * top_k, device=DEVICE)
    y = torch.zeros(t, n, dtype=torch.float64, device=DEVICE)
    for j in range(top_k):
        y += weights[:, j:j + 1] * y_permuted[position.view(t, top_k)[:, j]]
    out["y"] = y
    return out
