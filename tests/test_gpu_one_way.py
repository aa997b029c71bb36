"""Counts of one-way patterns (every entry's row above its column, none of the
transposes): 1,500 of 6,000 vertices occur as columns only, so their lists are
empty and their sums zero, and the vertices above them read those sums."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U3 = [(0, 1), (1, 2)]
U5 = [(0, 1), (1, 2), (2, 3), (3, 4)]
TREE7 = [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]
TREE10 = [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]
PATH12 = [(i, i + 1) for i in range(11)]
N, EMPTY = 6000, 1500


@pytest.fixture(scope="module")
def one_way():
    """(colptr, rowidx): random pairs, the lower number the column, rows from
    1,500 on, and a vertex of 700 entries, above the default hub degree."""
    rng = np.random.default_rng(83)
    a, b = rng.integers(0, N - 1, 240000), rng.integers(EMPTY, N - 1, 240000)
    cols = np.concatenate([a[a < b], rng.choice(N - 1, 700, replace=False)])
    rows = np.concatenate([b[a < b], np.full(700, N - 1)])
    pairs = np.unique(np.stack([cols, rows], 1), axis=0)
    colptr = np.concatenate([[0], np.cumsum(np.bincount(pairs[:, 0], minlength=N))]).astype(np.int32)
    rowidx = np.ascontiguousarray(pairs[:, 1], np.int32)
    assert np.all(np.diff(colptr)[:EMPTY] > 0)  # active, though their lists are empty
    return colptr, rowidx


def _check(ctx, graph, order, k, edges, colorings, precision, hub_degree=512):
    """FP32 counts equal the oracle's restatement of the reference, FP64 ones its
    FP64 counts, up to the order of the final sum: below 6,000 terms, none
    negative, 6,000 * 2^-53 < 1e-12 relative (and FP64 tables the same again a
    step, 700 * 2^-53).  Before each count the symmetric pattern of the same pairs
    is counted in the same buffers, which leaves sums where the empty lists' are."""
    colptr, rowidx = graph
    keys = ("vertex_order", "hub_degree")
    saved = [ctx.get_option(key) for key in keys]
    try:
        ctx.set_option("hub_degree", hub_degree)
        ctx.set_option("vertex_order", order)
        lower = np.repeat(np.arange(N, dtype=np.int32), np.diff(colptr))
        symmetric = sg.csc_from_edges(N, lower, rowidx)
        plan = ctx.plan(k, edges)
        op = oracle.Plan(k, edges)
        rng = np.random.default_rng(89 + k)
        ref = oracle.count_f32 if precision == "fp32" else oracle.count_f64
        for B in colorings:
            cols = rng.integers(0, k, size=(B, N)).astype(np.uint8)
            print(f"[one way] k={k} B={B} order={order} {precision}", flush=True)
            ctx.upload_graph(*symmetric)
            ctx.count(plan, B, colors=cols, precision=precision)
            ctx.upload_graph(colptr, rowidx)
            got = ctx.count(plan, B, colors=cols, precision=precision)
            for i in range(B):
                want = ref(op, colptr, rowidx, cols[i])
                assert abs(got[i] - want) <= 1e-12 * abs(want), (B, i, got[i], want)
    finally:
        for key, v in zip(keys, saved):
            ctx.set_option(key, v)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("order", [0, 1])
def test_roots_of_empty_lists(gpu_ctx, one_way, order, precision):
    """A root with a leaf main child, by tiles: one coloring, four, and a pass too
    wide for them."""
    _check(gpu_ctx, one_way, order, 3, U3, (1, 4, 5), precision)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("k,edges,colorings", [
    (5, U5, (1, 5, 16)),     # streamed rows of 4 and 6 values
    (7, TREE7, (1, 5)),      # rows of 15 and 20
    (10, TREE10, (1, 8)),    # a combine of its own: Y in the output's unwritten rows
    (12, PATH12, (2,)),      # whole rows and lanes beside the streamed ones
])
def test_sums_of_empty_lists(gpu_ctx, one_way, k, edges, colorings, order, precision):
    # (FP64 rows are streamed where the hubs hold a quarter of the entries)
    _check(gpu_ctx, one_way, order, k, edges, colorings, precision, 512 if precision == "fp32" else 31)
