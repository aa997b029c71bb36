"""The hubs that 16 wavefronts share are a prefix of the internal order under
either vertex order, also where the breadth-first one meets smaller hubs first."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U3 = [(0, 1), (1, 2)]
DEGREES = (9000, 2000, 1500, 5000, 1100, 4097, 4096)  # three above 4,096


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1])
def test_the_largest_hubs_come_first(gpu_ctx, order):
    """FP64 counts are whole numbers below 2^53: equal to the oracle's."""
    rng = np.random.default_rng(97)
    n, hubs = 12000, len(DEGREES)
    s, d = [], []
    for h, deg in enumerate(DEGREES):
        # all hubs are neighbours of the first: a breadth-first order takes them as numbered
        links = np.arange(1, hubs) if h == 0 else np.array([0])
        s.append(np.full(deg - len(links), h))
        d.append(rng.choice(np.arange(hubs, n), size=deg - len(links), replace=False))
    s.append(np.zeros(hubs - 1, int))
    d.append(np.arange(1, hubs))
    colptr, rowidx = sg.csc_from_edges(n, np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32))
    assert tuple(np.diff(colptr)[:hubs]) == DEGREES
    saved = gpu_ctx.get_option("vertex_order")
    try:
        gpu_ctx.set_option("vertex_order", order)
        gpu_ctx.upload_graph(colptr, rowidx)
        assert gpu_ctx.get_option("big_hubs") == 3
        cols = rng.integers(0, 3, size=(2, n)).astype(np.uint8)
        got = gpu_ctx.count(gpu_ctx.plan(3, U3), 2, colors=cols, precision="fp64")
        op = oracle.Plan(3, U3)
        assert got.tolist() == [oracle.count_f64(op, colptr, rowidx, c) for c in cols]
    finally:
        gpu_ctx.set_option("vertex_order", saved)
