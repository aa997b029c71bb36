"""Counts of one-way patterns (every entry's row above its column, none of the
transposes): 1,500 of 6,000 vertices occur as columns only, so their lists are
empty and their sums zero, and the vertices above them read those sums."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U3 = [(0, 1), (1, 2)]
N, EMPTY = 6000, 1500


@pytest.fixture(scope="module")
def one_way():
    """(colptr, rowidx): random pairs, the lower number the column, rows from
    1,500 on, and a vertex of 700 entries, above the default hub degree."""
    rng = np.random.default_rng(83)
    a, b = rng.integers(0, N - 1, 60000), rng.integers(EMPTY, N - 1, 60000)
    cols = np.concatenate([a[a < b], rng.choice(N - 1, 700, replace=False)])
    rows = np.concatenate([b[a < b], np.full(700, N - 1)])
    pairs = np.unique(np.stack([cols, rows], 1), axis=0)
    colptr = np.concatenate([[0], np.cumsum(np.bincount(pairs[:, 0], minlength=N))]).astype(np.int32)
    rowidx = np.ascontiguousarray(pairs[:, 1], np.int32)
    assert np.all(np.diff(colptr)[:EMPTY] > 0)  # active, though their lists are empty
    return colptr, rowidx


def _check(ctx, graph, order, k, edges, colorings, precision):
    """FP32 counts equal the oracle's restatement of the reference, FP64 ones its
    FP64 counts, up to the order of the final sum: below 6,000 terms, none
    negative, 6,000 * 2^-53 < 1e-12 relative (and FP64 tables the same again a
    step, 700 * 2^-53).  Other counts run first, so that the pass's buffers hold
    values of their own."""
    colptr, rowidx = graph
    saved = ctx.get_option("vertex_order")
    try:
        dense = sg.csc_from_edges(N, *(x.astype(np.int32) for x in np.triu_indices(120, 1)))
        plan = ctx.plan(k, edges)
        ctx.upload_graph(*dense)
        ctx.count(plan, max(colorings), seed=5, precision=precision)
        ctx.set_option("vertex_order", order)
        ctx.upload_graph(colptr, rowidx)
        op = oracle.Plan(k, edges)
        rng = np.random.default_rng(89 + k)
        ref = oracle.count_f32 if precision == "fp32" else oracle.count_f64
        for B in colorings:
            cols = rng.integers(0, k, size=(B, N)).astype(np.uint8)
            print(f"[one way] k={k} B={B} order={order} {precision}", flush=True)
            got = ctx.count(plan, B, colors=cols, precision=precision)
            for i in range(B):
                want = ref(op, colptr, rowidx, cols[i])
                assert abs(got[i] - want) <= 1e-12 * abs(want), (B, i, got[i], want)
    finally:
        ctx.set_option("vertex_order", saved)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("order", [0, 1])
def test_roots_of_empty_lists(gpu_ctx, one_way, order, precision):
    """A root with a leaf main child, by tiles: one coloring, four, and a pass too
    wide for them."""
    _check(gpu_ctx, one_way, order, 3, U3, (1, 4, 5), precision)
