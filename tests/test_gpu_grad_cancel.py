"""Gradients of colorings whose cotangents cancel: each coloring's part reaches
an entry's FP64 gradient with no FP32 sum over several colorings, in the steps
of wide dY rows by lanes (12 vertices, aux children of 3: rows of 165 values)."""
import numpy as np
import pytest

import subgraph_amd as sg

# three steps with an aux child of 3 vertices; every other aux child is a leaf
THREES = [(0, 1), (1, 2), (1, 3), (0, 4), (4, 5), (4, 6), (0, 7), (7, 8), (7, 9), (0, 10), (0, 11)]


@pytest.mark.gpu
@pytest.mark.parametrize("hub_degree", [16, 512])
@pytest.mark.parametrize("weighted", [False, True])
def test_opposite_cotangents_cancel(gpu_ctx, weighted, hub_degree):
    """Colorings that come twice, with cotangents c and -c: FP32 arithmetic is
    symmetric in sign, so a lane's parts are exact opposites and what is left are
    the roundings of FP64 sums: of at most 64 lanes and a few dozen adds an entry,
    of parts that add up to twice the gradient of one of each (all non-negative):
    below 256 * 2^-53 < 1e-13 of it."""
    n = 1 << 12
    colptr, rowidx = sg.csc_from_edges(n, *sg.rmat_edges(12, 8, seed=3))
    rng = np.random.default_rng(101)
    cols = rng.integers(0, 12, size=(2, n)).astype(np.uint8)
    saved = gpu_ctx.get_option("hub_degree")
    try:
        gpu_ctx.set_option("hub_degree", hub_degree)
        gpu_ctx.upload_graph(colptr, rowidx)
        if weighted:
            gpu_ctx.set_weights(rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32))
        plan = gpu_ctx.plan(12, THREES)
        _, one = gpu_ctx.count_grad(plan, 2, colors=cols, precision="fp32")
        _, left = gpu_ctx.count_grad(plan, 4, colors=np.repeat(cols, 2, axis=0), precision="fp32",
                                     cotangent=np.array([1.0, -1.0, 1.0, -1.0]))
        assert gpu_ctx.get_option("last_tile") == 4 and one.max() > 0
        assert np.all(np.abs(left) <= 1e-13 * one), np.abs(left / one)[one > 0].max()
    finally:
        gpu_ctx.set_weights(None)
        gpu_ctx.set_option("hub_degree", saved)
