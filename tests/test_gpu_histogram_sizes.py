"""histogram and histogram_exclusive_scan around the sizes where the kernel
changes (24576 routes below 32 experts, 49152 below 128, 65536 from there), with ids that crowd
one expert (counted with ballots), ragged tails of the id quads, ids off 16
bytes and ids outside [0, E): counts and offsets are whole numbers and exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import raggedroute_amd as rr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,routes", [
    (8, 1), (8, 3), (31, 24575), (31, 24576), (31, 24577), (32, 24577), (64, 4097), (256, 16387),
    (1000, 8191), (32, 49151), (64, 49152), (64, 49153), (1024, 49152), (127, 49153), (128, 65536), (128, 65537), (2, 20000),
])
@pytest.mark.parametrize("kind", ["uniform", "hot", "one", "two", "invalid"])
def test_counts_and_offsets(ctx, device, experts, routes, kind):
    rng = np.random.default_rng(experts + routes)
    ids = rng.integers(0, experts, routes)
    if kind == "hot":
        ids = np.where(rng.random(routes) < 0.5, experts - 1, ids)
    elif kind == "one":
        ids[:] = experts // 2
    elif kind == "two":
        ids = np.where(np.arange(routes) % 2 == 0, 0, experts - 1)
    elif kind == "invalid":
        ids = np.where(rng.random(routes) < 0.3, rng.choice([-1, experts, 2 ** 31 - 1, -2 ** 31], routes), ids)
    want = np.bincount(ids[(ids >= 0) & (ids < experts)], minlength=experts).astype(np.int32)
    for offset in (0, 1):
        buf = torch.zeros(routes + offset, dtype=torch.int32, device=device)
        buf[offset:] = torch.from_numpy(ids.astype(np.int32)).to(device)
        counts = torch.full((experts,), -7, dtype=torch.int32, device=device)
        offsets = torch.full((experts + 1,), -7, dtype=torch.int32, device=device)
        p = buf.data_ptr() + 4 * offset
        status = rr.histogram(rr.HistogramArgs(expert_ids=p, counts=counts.data_ptr(), route_pairs=routes,
                                               experts=experts), ctx)
        assert status.ok(), status.message
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), want)
        counts.fill_(-7)
        status = rr.histogram_exclusive_scan(rr.HistogramExclusiveScanArgs(
            expert_ids=p, counts=counts.data_ptr(), offsets=offsets.data_ptr(), route_pairs=routes,
            experts=experts), ctx)
        assert status.ok(), status.message
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), want)
        assert np.array_equal(offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(want)]))
