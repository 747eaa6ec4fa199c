"""Chains of more routes than the one-launch strip kernel holds: route
preparation over counted chunks (from 8192 routes, up to 256 experts and 256
chunks) and the strip kernel's gathered form (16384 routes and more, N <= 128,
K <= 256), compared bit for bit with the operators run one by one and checked
against the oracle; ids outside [0, E) leave their rows untouched."""
from __future__ import annotations

import numpy as np
import pytest

import raggedroute_amd as rr
from raggedroute_amd import workloads
from test_gpu_chain import ChainRun, check_chain, run_stages
from test_gpu_route_chain import RouteChainRun, _stages, check_route_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,experts,top_k,hidden,output,dist", [
    (2100, 16, 8, 64, 64, "uniform"), (2100, 256, 8, 128, 100, "zipf"), (4097, 64, 4, 192, 96, "uniform"),
    (8200, 200, 2, 256, 128, "zipf"), (16500, 3, 1, 64, 8, "uniform"), (5500, 9, 3, 252, 64, "uniform"),
    (1024, 64, 8, 260, 20, "uniform"),    # exactly 8 chunks; tiled kernel
    (1025, 257, 8, 68, 12, "zipf"),       # past 256 experts
    (8195, 64, 33, 4, 4, "uniform"),      # more than 256 chunks
    (9000, 5, 2, 7, 9, "single_hot"),     # widths off four floats
])
@pytest.mark.parametrize("keep", [True, False])
def test_route_chain(ctx, device, tokens, experts, top_k, hidden, output, dist, keep):
    cfg = workloads.RouteChainConfig("large", tokens, experts, hidden, output, top_k, dist)
    inp = workloads.route_chain_inputs(cfg, seed=3)
    dev = RouteChainRun(cfg, inp, device, with_x_permuted=keep, with_inverse=keep).run(ctx)
    check_route_chain(cfg, inp, dev)
    if keep:
        ref = _stages(cfg, inp, device, ctx)
        for key in ("counts", "offsets", "route_pos", "sorted_route", "x_permuted", "y_permuted", "y"):
            assert np.array_equal(dev[key].view(np.uint32), ref[key].view(np.uint32)), f"{key} differs"


@pytest.mark.parametrize("kind,tokens,experts,hidden,output", [
    ("tokens", 8200, 64, 64, 64), ("logits", 8200, 100, 128, 128), ("tokens", 12000, 33, 256, 60),
    ("logits", 9001, 256, 96, 33), ("tokens", 4097, 256, 64, 132), ("logits", 4200, 1024, 32, 16),
])
def test_chain(ctx, device, kind, tokens, experts, hidden, output):
    cfg = workloads.ChainConfig("large", tokens, experts, hidden, output, from_tokens=kind == "tokens")
    inp = workloads.chain_inputs(cfg, seed=8)
    fused = ChainRun(cfg, inp, device).run(ctx)
    ref = run_stages(cfg, inp, device, ctx)
    for key in ("logits", "ids", "weights", "counts", "offsets", "route_pos", "sorted_route", "x_permuted",
                "y_permuted", "y"):
        assert np.array_equal(fused[key].view(np.uint32), ref[key].view(np.uint32)), f"{key} differs"
    check_chain(cfg, inp, fused, sample_tokens=np.arange(0, tokens, 41))


@pytest.mark.parametrize("hidden,output", [(64, 64), (260, 40)])
def test_ids_outside_the_experts(ctx, device, hidden, output):
    cfg = workloads.RouteChainConfig("invalid", 2500, 32, hidden, output, 8, "uniform")
    inp = workloads.route_chain_inputs(cfg, seed=5)
    rng = np.random.default_rng(1)
    bad = rng.random(inp["ids"].shape) < 0.2
    inp["ids"] = np.where(bad, rng.choice([-1, 32, 1 << 30], bad.shape), inp["ids"]).astype(np.int32)
    dev = RouteChainRun(cfg, inp, device).run(ctx)
    flat, ok = inp["ids"].reshape(-1), ~bad.reshape(-1)
    counts = np.bincount(flat[ok], minlength=32)
    offsets = np.concatenate([[0], np.cumsum(counts)])
    assert np.array_equal(dev["counts"], counts) and np.array_equal(dev["offsets"], offsets)
    order = np.argsort(flat[ok], kind="stable")
    routes = np.nonzero(ok)[0][order]
    want = np.full(flat.size, -1)
    want[routes] = np.arange(routes.size)
    assert np.array_equal(dev["route_pos"], want)
    assert np.array_equal(dev["x_permuted"][:routes.size], inp["x"][routes // 8])
    for key in ("x_permuted", "y_permuted"):  # no row is written for such a route
        assert np.isnan(dev[key][routes.size:]).all()
    w = inp["weights"].reshape(-1)
    y = np.zeros((cfg.tokens, output))
    for r in np.nonzero(ok)[0]:
        y[r // 8] += np.float64(w[r]) * dev["y_permuted"][want[r]].astype(np.float64)
    assert np.allclose(dev["y"], y, rtol=1e-5, atol=1e-5 * np.abs(y).max())
