"""The combine of rows whose Y is in memory: parts of the vertices whose Y lies
in the output table's later rows, the last ones fused, and (for the adjoint)
all at once; groups of 16 rows with a remainder; Y from the narrow rows' and
from the wide rows' gather."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

TREE10 = [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]
TREE12 = [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (2, 6), (6, 7), (7, 8), (6, 9), (9, 10), (10, 11)]


def _graph(n):
    rng = np.random.default_rng(n)
    a, b = rng.integers(0, n, 2 * n), rng.integers(0, n, 2 * n)
    b = np.where(rng.random(2 * n) < 0.1, b % 40, b)  # some hubs
    keep = a != b
    pairs = np.unique(np.stack([np.minimum(a[keep], b[keep]), np.maximum(a[keep], b[keep])], 1), axis=0)
    return sg.csc_from_edges(n, pairs[:, 0].astype(np.int32), pairs[:, 1].astype(np.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("k,edges,n,B", [
    (12, TREE12, 5003, 1),     # every step fused but the one of 11 -> 55 values
    (12, TREE12, 19001, 1),    # one part of it and a fused rest
    (12, TREE12, 18011, 4),    # both steps in several parts
    (10, TREE10, 30011, 5),
])
def test_combined_rows_keep_the_reference_arithmetic(gpu_ctx, k, edges, n, B):
    """FP32 counts equal the oracle's restatement of the reference up to the
    order of the final FP64 sum (n * 2^-53 < 4e-12 relative for a sum of
    non-negative terms).  FP32 gradients, whose forward pass keeps Y, agree in
    norm with FP64 ones, which take the gathers' own combine, to the roundings
    of non-negative FP32 sums: below 2e-5 by the square root of the terms of a
    chain of k steps (k * 60 * 2^-24 < 5e-5 at the worst, all of one sign)."""
    colptr, rowidx = _graph(n)
    rng = np.random.default_rng(61 + k)
    cols = rng.integers(0, k, size=(B, n)).astype(np.uint8)
    saved = gpu_ctx.get_option("exact_order")
    try:
        gpu_ctx.set_option("exact_order", 1)
        gpu_ctx.upload_graph(colptr, rowidx)
        plan = gpu_ctx.plan(k, edges)
        op = oracle.Plan(k, edges)
        print(f"[combine] k={k} n={n} B={B}", flush=True)
        got = gpu_ctx.count(plan, B, colors=cols, precision="fp32")
        for i in range(B):
            want = oracle.count_f32(op, colptr, rowidx, cols[i])
            assert abs(got[i] - want) <= 4e-12 * abs(want), (i, got[i], want)
        r32, g32 = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp32")
        r64, g64 = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp64")
        assert np.array_equal(r32, got)
        assert np.linalg.norm(g32 - g64) <= 5e-5 * np.linalg.norm(g64)
    finally:
        gpu_ctx.set_option("exact_order", saved)
