"""The dense GEMM of at most 128 columns for shapes past the strip kernel
(K > 256, or rows off 16 bytes), and the router + gate launch built on it:
edges of its strips (one, two and four a workgroup), 64-deep slices, quads and
column counts. The sums have the tiled kernel's order, so the results must have
its bits (RR_GEMM_TILE=small), and the fused gate the gate kernel's."""
from __future__ import annotations

import os

import numpy as np
import pytest
import torch

import raggedroute_amd as rr
from raggedroute_amd import workloads
from test_gpu_chain import ChainRun, check_chain, run_stages
from test_gpu_ops import NATIVE, gemm_ok, ok

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,offset", [
    (1, 4, 1, 0), (15, 5, 63, 0), (16, 7, 64, 1), (17, 64, 65, 0), (33, 63, 127, 0), (31, 65, 128, 1),
    (100, 128, 320, 0), (100, 127, 321, 3), (48, 100, 1023, 0), (20, 16, 257, 0),
    (8192 + 5, 64, 130, 1), (8192 + 31, 101, 260, 0),        # two strips a workgroup
    (16384 + 33, 60, 300, 0), (16384 + 63, 128, 259, 1),     # four
])
def test_bits_of_the_tiled_kernel(ctx, device, m, n, k, offset):
    rng = np.random.default_rng(m + n + k)
    a_h = rng.standard_normal((m, k)).astype(np.float32)
    b_h = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
    a = torch.empty(m * k + offset, device=device)
    b = torch.empty(k * n + offset, device=device)
    a[offset:] = torch.from_numpy(a_h.reshape(-1)).to(device)
    b[offset:] = torch.from_numpy(b_h.reshape(-1)).to(device)

    def run():
        c = torch.full((m * n + 64,), 7.0, device=device)
        ok(rr.dense_gemm(rr.DenseGemmArgs(a=rr.cview(a.data_ptr() + 4 * offset), b=rr.cview(b.data_ptr() + 4 * offset),
                                          c=rr.mview(c.data_ptr()), m=m, n=n, k=k, kernel=NATIVE), ctx))
        torch.cuda.synchronize()
        assert (c[m * n:] == 7.0).all()
        return c[:m * n].cpu().numpy().reshape(m, n)
    got = run()
    saved = os.environ.get("RR_GEMM_TILE")
    os.environ["RR_GEMM_TILE"] = "small"
    try:
        want = run()
    finally:
        os.environ.pop("RR_GEMM_TILE")
        if saved is not None:
            os.environ["RR_GEMM_TILE"] = saved
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    gemm_ok(got[:64], a_h[:64], b_h)


@pytest.mark.parametrize("tokens,experts,hidden,output", [
    (5, 4, 257, 8), (100, 64, 300, 33), (77, 65, 511, 20), (333, 128, 260, 7), (8192 + 9, 7, 270, 12),
    (16384 + 17, 100, 258, 5),
])
def test_router_and_gate_launch(ctx, device, tokens, experts, hidden, output):
    cfg = workloads.ChainConfig("router", tokens, experts, hidden, output)
    inp = workloads.chain_inputs(cfg, seed=9)
    fused = ChainRun(cfg, inp, device).run(ctx)
    ref = run_stages(cfg, inp, device, ctx)
    for key in ("logits", "ids", "weights", "counts", "offsets", "route_pos", "x_permuted", "y_permuted", "y"):
        assert np.array_equal(fused[key].view(np.uint32), ref[key].view(np.uint32)), f"{key} differs"
    check_chain(cfg, inp, fused, sample_tokens=np.arange(0, tokens, max(1, tokens // 200)))
