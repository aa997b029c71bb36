"""The neighbours' colours of an entry, written 16, 8, 4 bytes of one entry or
four bytes of several at a time: each number of colorings in one pass gives
the counts and gradients of the same colorings one by one."""
import numpy as np
import pytest

import subgraph_amd as sg

U4 = [(0, 1), (1, 2), (1, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize("B", [2, 3, 4, 5, 6, 7, 8, 12, 16, 24, 32, 33])
def test_colorings_of_a_pass_equal_single_ones(gpu_ctx, B):
    """An odd number of undirected edges, so that a pass of an odd number of
    colorings ends within a word.  FP64 values are integers below 2^53: equal;
    a pass's gradient is the sum of its colorings'."""
    rng = np.random.default_rng(67)
    n = 700
    a, b = rng.integers(0, n, 4000), rng.integers(0, n, 4000)
    pairs = np.unique(np.stack([np.minimum(a, b), np.maximum(a, b)], 1)[a != b], axis=0)
    pairs = pairs[:len(pairs) - (len(pairs) + 1) % 2]
    colptr, rowidx = sg.csc_from_edges(n, pairs[:, 0].astype(np.int32), pairs[:, 1].astype(np.int32))
    assert len(rowidx) % 4 == 2
    gpu_ctx.upload_graph(colptr, rowidx)
    gpu_ctx.set_weights(None)
    plan = gpu_ctx.plan(4, U4)
    cols = rng.integers(0, 4, size=(B, n)).astype(np.uint8)
    print(f"[edge colors] B={B}", flush=True)
    got = gpu_ctx.count(plan, B, colors=cols, precision="fp64")
    _, grad = gpu_ctx.count_grad(plan, B, colors=cols, precision="fp64")
    want_grad = np.zeros(len(rowidx))
    for i in range(B):
        assert got[i] == gpu_ctx.count(plan, 1, colors=cols[i:i + 1], precision="fp64")[0]
        want_grad += gpu_ctx.count_grad(plan, 1, colors=cols[i:i + 1], precision="fp64")[1]
    assert np.array_equal(grad, want_grad)
