"""The streamed sums of narrow rows where they can go wrong: lists that end at
and around a batch of 48 entries, tiles closed by their entries (256), by their
vertices (256), and of one longer list; rows of 1 to 63 values, as many
colorings as a wavefront takes and one more; weights; a scaled first step."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U5 = [(0, 1), (1, 2), (2, 3), (3, 4)]
TREE7 = [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]
TREE10 = [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]
PATH12 = [(i, i + 1) for i in range(11)]
# list lengths of the vertices that are not hubs (hub_degree 4096 below)
LENGTHS = (1, 2, 46, 47, 48, 49, 95, 96, 97, 207, 208, 209, 255, 256, 257, 300, 1500)


def _graph():
    """A vertex of every length, and 700 of one neighbour each (tiles closed by
    their vertices), over 6,000 vertices that a sparse random graph links."""
    rng = np.random.default_rng(53)
    own = len(LENGTHS)
    n = own + 6000 + 700
    s, d = [], []
    for v, deg in enumerate(LENGTHS):
        s.append(np.full(deg, v))
        d.append(rng.choice(np.arange(own, own + 6000), size=deg, replace=False))
    s.append(np.arange(own + 6000, n))
    d.append(rng.integers(own, own + 6000, 700))
    a, b = rng.integers(own, own + 6000, 9000), rng.integers(own, own + 6000, 9000)
    keep = a != b
    pairs = np.unique(np.stack([np.minimum(a[keep], b[keep]), np.maximum(a[keep], b[keep])], 1), axis=0)
    s.append(pairs[:, 0])
    d.append(pairs[:, 1])
    colptr, rowidx = sg.csc_from_edges(n, np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32))
    assert tuple(np.diff(colptr)[:own]) == LENGTHS
    return n, colptr, rowidx


@pytest.mark.gpu
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("k,edges,colorings", [
    (5, U5, (1, 3, 10, 11, 33)),   # rows of 6 (10 colorings a wavefront) and 4 values
    (7, TREE7, (1, 3, 4)),         # rows of 15 and 20 values, 3 colorings
    (10, TREE10, (1, 7)),          # rows of 36 into 9, one coloring
    (12, PATH12, (1, 5, 6)),       # rows of 12 and less into wider ones
])
def test_streamed_rows_keep_the_reference_arithmetic(gpu_ctx, k, edges, colorings, weighted):
    """FP32 counts equal the oracle's restatement of the reference up to the
    order of the final FP64 sum over n < 7,000 vertices (7,000 * 2^-53 < 1e-12
    relative for a sum of non-negative terms).  Weighted ones equal its FP64
    counts up to FP32 rounding: of at most 1,500 products and additions a step,
    and the combine's few, all non-negative."""
    n, colptr, rowidx = _graph()
    keys = ("hub_degree", "exact_order")
    saved = [gpu_ctx.get_option(key) for key in keys]
    try:
        gpu_ctx.set_option("hub_degree", 4096)
        gpu_ctx.set_option("exact_order", 1)
        gpu_ctx.upload_graph(colptr, rowidx)
        rng = np.random.default_rng(59 + k)
        weights = rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32) if weighted else None
        gpu_ctx.set_weights(weights)
        plan = gpu_ctx.plan(k, edges)
        op = oracle.Plan(k, edges)
        for B in colorings:
            cols = rng.integers(0, k, size=(B, n)).astype(np.uint8)
            print(f"[stream] k={k} B={B}", flush=True)
            got = gpu_ctx.count(plan, B, colors=cols, precision="fp32")
            for i in range(B):
                if weighted:
                    want, tol = oracle.count_f64(op, colptr, rowidx, cols[i], vals=weights), (k - 1) * 1510 * 2.0**-24
                else:
                    want, tol = oracle.count_f32(op, colptr, rowidx, cols[i]), 1e-12
                assert abs(got[i] - want) <= tol * abs(want), (B, i, got[i], want)
    finally:
        gpu_ctx.set_weights(None)
        for key, v in zip(keys, saved):
            gpu_ctx.set_option(key, v)


@pytest.mark.gpu
@pytest.mark.parametrize("hub_degree", [64, 4096])
@pytest.mark.parametrize("k,edges,colorings", [
    (5, U5, (12, 33)),       # rows of 4 into 6 values and of 1 into 4, two and more chunks
    (12, PATH12, (1, 4)),    # rows of 11 into 55, a coloring a chunk
])
def test_streamed_gradients_of_every_entry(gpu_ctx, k, edges, colorings, hub_degree):
    """FP32 gradients of weighted counts equal the FP64 ones, entry by entry, up
    to FP32 rounding: of at most 1,500 products and additions a step forward and
    as many backward, all non-negative."""
    n, colptr, rowidx = _graph()
    saved = gpu_ctx.get_option("hub_degree")
    try:
        gpu_ctx.set_option("hub_degree", hub_degree)
        gpu_ctx.upload_graph(colptr, rowidx)
        rng = np.random.default_rng(71 + k)
        gpu_ctx.set_weights(rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32))
        plan = gpu_ctx.plan(k, edges)
        tol = 2 * (k - 1) * 1510 * 2.0**-24
        for B in colorings:
            cols = rng.integers(0, k, size=(B, n)).astype(np.uint8)
            print(f"[stream grad] k={k} B={B} hub_degree={hub_degree}", flush=True)
            _, g32 = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp32")
            _, g64 = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp64")
            assert np.all(np.abs(g32 - g64) <= tol * np.abs(g64)), np.abs(g32 / g64 - 1)[g64 > 0].max()
    finally:
        gpu_ctx.set_weights(None)
        gpu_ctx.set_option("hub_degree", saved)
