"""The streamed sums of narrow FP64 rows where they can go wrong: lists that end
at and around a batch of 32 entries, tiles closed by their entries, by their
vertices and of one longer list, rows of 4 to 55 values, as many colorings as a
wavefront takes and one more, on a graph whose hubs hold a quarter of the
entries (without that these rows are not streamed)."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U5 = [(0, 1), (1, 2), (2, 3), (3, 4)]
TREE7 = [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]
PATH12 = [(i, i + 1) for i in range(11)]
LENGTHS = (1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 255, 256, 257, 300, 1700, 1700, 1700, 1700)


def _graph():
    rng = np.random.default_rng(61)
    own, n = len(LENGTHS), len(LENGTHS) + 3000
    s = [np.full(deg, v) for v, deg in enumerate(LENGTHS)]
    d = [rng.choice(np.arange(own, own + 2000), size=deg, replace=False) for deg in LENGTHS]
    s.append(np.arange(own + 2000, n))
    d.append(rng.integers(own, own + 2000, 1000))
    a, b = rng.integers(own, own + 2000, 3000), rng.integers(own, own + 2000, 3000)
    pairs = np.unique(np.stack([np.minimum(a, b), np.maximum(a, b)], 1)[a != b], axis=0)
    s.append(pairs[:, 0])
    d.append(pairs[:, 1])
    colptr, rowidx = sg.csc_from_edges(n, np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32))
    assert tuple(np.diff(colptr)[:own]) == LENGTHS
    assert 4 * 1700 >= len(rowidx) / 4
    return n, colptr, rowidx


@pytest.mark.gpu
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("hub_degree", [64, 1024])
@pytest.mark.parametrize("k,edges,colorings", [
    (5, U5, (1, 10, 11, 33)),   # rows of 6 and 4 values: 10 colorings a wavefront
    (7, TREE7, (1, 3, 4)),      # 15 and 20 values: 3 colorings
    (12, PATH12, (1, 5)),       # 11 into 55
])
def test_streamed_fp64_rows(gpu_ctx, k, edges, colorings, hub_degree, weighted):
    """FP64 counts equal the oracle's up to the rounding of at most 1,710 products
    and additions a step and the final sum over n < 3,100 vertices, all
    non-negative; the gradients equal those of the separate gathers (fuse_grad
    0), entry by entry, up to that rounding forward and backward, and satisfy
    sum_e w_e grad_e = (k - 1) * count."""
    n, colptr, rowidx = _graph()
    keys = ("hub_degree", "hub_chunk", "exact_order", "fuse_grad")
    saved = [gpu_ctx.get_option(key) for key in keys]
    try:
        gpu_ctx.set_option("hub_degree", hub_degree)
        gpu_ctx.set_option("hub_chunk", 33)
        gpu_ctx.set_option("exact_order", 1)
        gpu_ctx.upload_graph(colptr, rowidx)
        rng = np.random.default_rng(67 + k)
        w = rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32) if weighted else None
        gpu_ctx.set_weights(w)
        plan = gpu_ctx.plan(k, edges)
        op = oracle.Plan(k, edges)
        tol = ((k - 1) * 1710 + 3100) * 2.0**-52
        for B in colorings:
            cols = rng.integers(0, k, size=(B, n)).astype(np.uint8)
            print(f"[stream64] k={k} B={B} hub_degree={hub_degree} weighted={weighted}", flush=True)
            got = gpu_ctx.count(plan, B, colors=cols, precision="fp64")
            for i in range(B):
                want = oracle.count_f64(op, colptr, rowidx, cols[i], vals=w)
                assert abs(got[i] - want) <= tol * abs(want), (B, i, got[i], want)
            grads = {}
            for fuse in (1, 0):
                gpu_ctx.set_option("fuse_grad", fuse)
                raw, grads[fuse] = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp64")
            assert np.all(np.abs(grads[1] - grads[0]) <= 2 * B * tol * np.abs(grads[0]))
            ww = np.ones(len(rowidx)) if w is None else w.astype(np.float64)
            total = (k - 1) * raw.sum()
            assert abs((grads[1] * ww).sum() - total) <= 2 * (tol * B + len(rowidx) * 2.0**-52) * abs(total)
    finally:
        gpu_ctx.set_weights(None)
        for key, v in zip(keys, saved):
            gpu_ctx.set_option(key, v)
