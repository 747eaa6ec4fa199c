"""The grouped GEMM on the BF16 matrix cores, forced into each of its workgroup
shapes with RR_GEMM_STAGING=split4 (four waves, 128-row tiles), split8 (eight)
and split256 (eight, 256-row tiles): row counts at the edges of its 32-row blocks
and tiles, K and N at the edges of its slices, pairs and column tiles, offset
pointers, and values of every range (infinities, NaN, overflow, subnormals,
outliers either way). Outputs that are not finite, or below 2^-80, must be the FP32
instructions' (RR_GEMM_STAGING=fp32).

Tolerances: check_grouped's accumulation-aware bound 4 gamma_K sum |a b| + 1e-7
of the float64 product for every output, and, since that grows with K where the
split's own error does not, a 2-norm bound: the three parts hold every bit, the
products left out are 2^-25 of one, and the large sum rounds once per 16 k: under
the FP32 instructions' error sqrt(K) 2^-26 for K >= 64. A lost or misplaced part shows
as 2^-9 or 2^-17 of a product, 20 times that and more.
"""
from __future__ import annotations

import os

import numpy as np
import pytest

import raggedroute_amd as rr
from raggedroute_amd import workloads
from test_gpu_chain import ChainRun, check_chain, run_stages
from test_gpu_ops import NATIVE, check_grouped, run_grouped

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def staging():
    saved = os.environ.get("RR_GEMM_STAGING")

    def put(name):
        os.environ["RR_GEMM_STAGING"] = name
    put("split")
    yield put
    os.environ.pop("RR_GEMM_STAGING", None)
    if saved is not None:
        os.environ["RR_GEMM_STAGING"] = saved


EDGE_ROWS = [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 192, 193, 255, 256, 257]
SHAPES = ["split4", "split8", "split256"]


def two_norm_error(y, x, w, offsets):
    num = den = 0.0
    for e in range(len(w)):
        rows = slice(int(offsets[e]), int(offsets[e + 1]))
        exact = x[rows].astype(np.float64) @ w[e].astype(np.float64)
        num += ((y[rows] - exact) ** 2).sum()
        den += (exact ** 2).sum()
    return np.sqrt(num / den)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("counts,k,n,offset", [
    (EDGE_ROWS, 256, 272, 0),
    (EDGE_ROWS, 257, 273, 0),              # one float in the last slice, odd N: the last pair is half a pair
    (EDGE_ROWS[::-1], 287, 383, 1),        # pointers off 16 bytes
    ([5, 0, 200, 70], 288, 384, 0),        # whole slices, whole column tiles
    ([5, 0, 200, 70], 319, 385, 3),        # a column tile of one column
    ([300, 40, 129], 1023, 641, 0),
    ([9] * 130, 256, 300, 0),              # more tiles than workgroups per XCD
    ([3] * 1024, 256, 272, 0),             # E = 1024
    (EDGE_ROWS, 130, 1701, 1),
    # more tiles than workgroups in every shape, 256-row tiles at their layouts' edges
    ([513, 700, 767, 1, 300, 1100], 163, 3301, 1),
    ([513, 447, 448, 576, 640, 832], 160, 3328, 0),
    ([70, 3], 1, 2, 0),                    # one float, one pair
    ([70, 3], 33, 5, 1),                   # two slices
    ([70, 3], 65, 131, 0),                 # three slices
    # one slice to eight, whole and not: the ends of the loops of one and of two slices a turn
    *[([70, 3], k, 132, 0) for k in (16, 17, 32, 48, 64, 80, 96, 111, 112, 128)],
])
def test_edges(ctx, device, staging, shape, counts, k, n, offset):
    staging(shape)
    rng = np.random.default_rng(sum(counts) + k + n)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    rows = int(offsets[-1])
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (rng.standard_normal((len(counts), k, n)) / np.sqrt(k)).astype(np.float32)
    y = run_grouped(ctx, device, x, w, offsets, NATIVE, max_tokens=max(counts), offset=offset, rows_total=rows)
    check_grouped(y, x, w, offsets)
    # (sqrt(64) below K = 64; 1.5 for few outputs)
    assert two_norm_error(y, x, w, offsets) <= 1.5 * np.sqrt(max(k, 64)) * 2.0 ** -26


def special_inputs(case, rng):
    counts, k, n = [200, 40, 90, 20], 320, 400
    x = rng.standard_normal((sum(counts), k)).astype(np.float32)
    w = (rng.standard_normal((4, k, n)) / np.sqrt(k)).astype(np.float32)
    if case == "infinity and NaN":
        x[3, 100] = np.inf
        x[210, 5] = np.nan
        w[2, 7, 9] = -np.inf
    elif case == "late outlier":
        x[:, 200] *= 1e6
    elif case == "early outlier":     # 2^20 times the rest, and weights that do not meet it
        x[:, :32] *= 2.0 ** 20
        w[:, :32] = 0
    elif case == "early outliers of both":  # 2^10, in separate columns
        x[:, :16] *= 2.0 ** 10
        w[:, :16] = 0
        w[:, 16:32] *= 2.0 ** 10
        x[:, 16:32] = 0
    elif case == "zeros":             # zero rows, zero columns, leading zeros of both
        x[7] = 0
        x[:, :64] = 0
        x[220] = 0
        w[:, :100] = 0
        w[1, :, 7] = 0
    elif case == "all zero":
        x[:] = 0
    elif case == "tiny":
        x *= np.float32(1e-34)
    elif case == "subnormal":
        x *= np.float32(1e-38)
        w *= np.float32(1e3)
    elif case == "huge":
        x *= np.float32(1e37)
        w *= np.float32(1e-5)
    elif case == "overflow":          # the first rows' sums pass the FP32 range, whatever their order
        x[:100] = np.minimum(np.abs(x[:100]), 1.5) * np.float32(2e38)
        w = np.abs(w)
    elif case == "row scales":
        x *= np.logspace(-18, 18, x.shape[0], dtype=np.float32)[:, None]
        w *= np.logspace(-9, 9, n, dtype=np.float32)
    return counts, x, w


@pytest.mark.parametrize("case", ["infinity and NaN", "late outlier", "early outlier", "early outliers of both",
                                  "zeros", "all zero", "tiny", "subnormal",
                                  "huge", "overflow", "row scales"])
@pytest.mark.parametrize("shape", SHAPES)
def test_values_of_every_range(ctx, device, staging, shape, case):
    counts, x, w = special_inputs(case, np.random.default_rng(11))
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    staging("fp32")
    want = run_grouped(ctx, device, x, w, offsets, NATIVE)
    staging(shape)
    got = run_grouped(ctx, device, x, w, offsets, NATIVE)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    # the finite ones: both lie within 4 gamma_K sum |a b| of the exact sums
    # (and a few subnormal steps: each product and sum may round to one)
    gamma = x.shape[1] * 2.0 ** -24
    with np.errstate(over="ignore", invalid="ignore"):
        for e, c in enumerate(counts):
            s = int(offsets[e])
            mag = np.abs(x[s:s + c].astype(np.float64)) @ np.abs(w[e].astype(np.float64))
            exact = x[s:s + c].astype(np.float64) @ w[e].astype(np.float64)
            fin = np.isfinite(want[s:s + c])
            err = np.abs(got[s:s + c].astype(np.float64) - exact)
            assert (err <= 4 * gamma * mag + 2 * x.shape[1] * 2.0 ** -149)[fin].all(), (case, e)


@pytest.mark.parametrize("path,experts,rows,k,n", [
    # few rows an expert, many tiles; few tiles; short K
    ("fp32", 64, 256, 128, 1024), ("fp32", 64, 1024, 256, 1024), ("fp32", 32, 128, 1024, 2048),
    ("fp32", 8, 32, 512, 2048), ("fp32", 8, 1024, 1024, 512), ("fp32", 16, 1600, 128, 1024),
    # enough of both
    ("split", 64, 3072, 128, 1024), ("split", 32, 512, 512, 500), ("split", 8, 4096, 1024, 512),
    ("split", 16, 1600, 192, 1024), ("split", 8, 1200, 256, 1536),
])
def test_kernel_by_size(ctx, device, staging, path, experts, rows, k, n):
    """The kernel that measures faster on MI355X (256 CUs), seen by its bits."""
    rng = np.random.default_rng(rows + k)
    counts = np.bincount(rng.integers(0, experts, rows), minlength=experts)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (rng.standard_normal((experts, k, n)) / np.sqrt(k)).astype(np.float32)
    y = {}
    for name in ("fp32", "split", "default"):
        staging(name)
        y[name] = run_grouped(ctx, device, x, w, offsets, NATIVE)
    assert not np.array_equal(y["fp32"], y["split"])
    assert np.array_equal(y["default"], y[path])


@pytest.mark.parametrize("case", ["infinity and NaN", "late outlier", "tiny", "subnormal", "overflow", "row scales", "scattered"])
def test_outputs_depend_on_their_row_and_column_only(ctx, device, staging, case):
    """Each output is the split's or, not finite or below 2^-80, the FP32 kernels' bit
    for bit, by its own value: the same in every workgroup shape (so whatever other
    rows its tile holds), and where rows or columns change, no other output moves."""
    if case == "scattered":  # a few odd rows and columns in tiles of ordinary ones
        rng = np.random.default_rng(12)
        counts, k, n = [700, 3, 257, 130], 200, 300
        x = rng.standard_normal((sum(counts), k)).astype(np.float32)
        w = (rng.standard_normal((4, k, n)) / np.sqrt(k)).astype(np.float32)
        plain = x.copy(), w.copy()
        rows, cols = [5, 300, 511, 800], {0: [7, 290], 2: [131]}
        x[5, 199] = np.inf
        x[300] *= np.float32(2.0 ** -100)
        x[511, 100] = 3e38
        x[800, 3] = np.nan
        for e, cs in cols.items():
            w[e][60, cs] = np.inf
    else:
        counts, x, w = special_inputs(case, np.random.default_rng(11))
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)

    def bits(path, xs, ws):
        staging(path)
        return run_grouped(ctx, device, xs, ws, offsets, NATIVE).view(np.uint32)
    fp32 = bits("fp32", x, w)
    split = [bits(shape, x, w) for shape in SHAPES]
    for other in split[1:]:
        assert np.array_equal(split[0], other)
    # (2^-81: the split's own value decides, an ulp beside this one)
    value = np.abs(fp32.view(np.float32))
    own = ~np.isfinite(value) | (value < 2.0 ** -81)
    assert np.array_equal(split[0][own], fp32[own])
    if case in ("tiny", "subnormal"):
        assert own.all()
    if case == "scattered":
        assert own[[5, 300, 800]].all()
        touched = np.zeros(fp32.shape, bool)
        touched[rows] = True
        for e, cs in cols.items():
            touched[offsets[e]:offsets[e + 1], cs] = True
        assert np.array_equal(split[0][~touched], bits("split4", *plain)[~touched])


@pytest.mark.parametrize("p", [-40, -20, -12, 0, 9, 11, 30])
@pytest.mark.parametrize("side", ["row", "column"])
def test_zero_first_slice(ctx, device, staging, side, p):
    """All-zero rows and columns, and ones whose first slice is zero and whose
    other values are 2^p: as close to the exact results as the FP32 instructions'
    (the bound of test_values_of_two_scales)."""
    rng = np.random.default_rng(p + 50)
    counts, k, n = [200, 40, 90, 20], 320, 400
    x = rng.standard_normal((sum(counts), k)).astype(np.float32)
    w = (rng.standard_normal((4, k, n)) / np.sqrt(k)).astype(np.float32)
    a = x.T if side == "row" else w.transpose(1, 0, 2)  # views, k first
    a *= np.float32(2.0 ** p)
    a[:32] = 0
    a[..., 5::17] = 0
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    y = {}
    for path in ("fp32", "split4", "split8", "split256"):
        staging(path)
        y[path] = run_grouped(ctx, device, x, w, offsets, NATIVE)
    assert np.array_equal(y["split4"], y["split8"]) and np.array_equal(y["split4"], y["split256"])
    assert two_norm_error(y["split4"], x, w, offsets) <= 1.25 * two_norm_error(y["fp32"], x, w, offsets)
    assert (y["split4"] == 0)[y["fp32"] == 0].all()


@pytest.mark.parametrize("shape", ["split4", "split8"])
def test_chain_with_odd_rows(ctx, device, staging, shape):
    """The chain's gathered form (128-row tiles) against the staged operators in
    256-row tiles, with rows in x whose outputs are recomputed: every output the
    same bits."""
    cfg = workloads.ChainConfig("split", 700, 5, 256, 272)
    inp = workloads.chain_inputs(cfg, seed=6)
    x = inp["x"]
    x[3, 100] = 3e38
    x[77, 255] = -4e6
    x[300] *= np.float32(2.0 ** -100)
    x[301, 200] = np.inf
    x[555] = 0
    staging(shape)
    fused = ChainRun(cfg, inp, device).run(ctx)
    staging("split256")
    ref = run_stages(cfg, inp, device, ctx)
    assert not np.isfinite(fused["y"]).all() and np.isfinite(fused["y"]).any()
    for key in ("ids", "route_pos", "x_permuted", "y_permuted", "y"):
        assert np.array_equal(fused[key].view(np.uint32), ref[key].view(np.uint32)), f"{key} differs"


@pytest.mark.parametrize("side", ["row", "column"])
@pytest.mark.parametrize("form", ["zero", "compensating", "alternating", "three of four", "first slices", "last slice",
                                  "all but one"])
@pytest.mark.parametrize("p", [16, 22, 24, 27, 30, 36, 45, 60, -20, -60])
def test_values_of_two_scales(ctx, device, staging, side, form, p):
    """Features 2^p times the rest, met by zeros or by values 2^-p the rest's: the
    results rest on the small ones alone, or on both. Either way they must be as
    close to the exact ones as the FP32 instructions' (whose error differs by the
    order of the sums only: a few percent over these 140000 outputs; 1.25 times
    is allowed)."""
    rng = np.random.default_rng(p + 100)
    counts, k, n = [200, 40, 90, 20], 320, 400
    big = {"zero": slice(0, 1), "compensating": slice(0, 1), "alternating": slice(0, None, 2),
           "three of four": np.arange(k) % 4 != 1, "first slices": slice(0, 96), "last slice": slice(0, 288), "all but one": np.arange(k) != 200}[form]
    x = rng.standard_normal((sum(counts), k)).astype(np.float32)
    w = (rng.standard_normal((4, k, n)) / np.sqrt(k)).astype(np.float32)
    a, b = (x.T, w.transpose(1, 0, 2)) if side == "row" else (w.transpose(1, 0, 2), x.T)  # views, k first
    a[big] *= np.float32(2.0 ** p)
    b[big] *= np.float32(2.0 ** -p if form == "compensating" else 0.0)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    err = {}
    for path in ("fp32", "split"):
        staging(path)
        err[path] = two_norm_error(run_grouped(ctx, device, x, w, offsets, NATIVE), x, w, offsets)
    assert err["split"] <= 1.25 * err["fp32"], err


@pytest.mark.parametrize("tokens,experts,hidden,output", [
    (700, 8, 256, 272), (333, 5, 289, 301), (64, 16, 512, 384), (1100, 7, 260, 640),
])
@pytest.mark.parametrize("shape", ["split4", "split8"])
def test_chain_form_matches_stage_by_stage(ctx, device, staging, shape, tokens, experts, hidden, output):
    staging(shape)
    cfg = workloads.ChainConfig("split", tokens, experts, hidden, output)
    inp = workloads.chain_inputs(cfg, seed=6)
    fused = ChainRun(cfg, inp, device).run(ctx)
    ref = run_stages(cfg, inp, device, ctx)
    for key in ("logits", "ids", "counts", "offsets", "route_pos", "x_permuted", "y_permuted", "y"):
        a, b = fused[key], ref[key]
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"{key} differs"
    check_chain(cfg, inp, fused)
