"""The hub kernel's neighbour lists at the lengths where it can go wrong:
around its batches of entries, around the turns of 4 and of 16 wavefronts, and
around the degree from which a hub takes a whole workgroup; rows narrower and
wider than a wavefront, one coloring per wavefront and several packed.  With
fewer hubs the same lists go through the other vertices' kernels: the root's
tiles (of 1,024 entries and 256 vertices, a longer list in windows) among them."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

TREE7 = [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]
TREE10 = [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]
U3 = [(0, 1), (1, 2)]
U5 = [(0, 1), (1, 2), (2, 3), (3, 4)]
PATH12 = [(i, i + 1) for i in range(11)]
STAR6 = [(0, 1), (1, 2), (1, 3), (1, 4), (1, 5)]
# list lengths: one batch (32 FP64, 56 FP32 entries) and its neighbours, whole
# rounds of 4 and 16 wavefronts, the whole-workgroup degree, a long list
LENGTHS = (17, 31, 32, 33, 55, 56, 57, 127, 128, 129, 223, 224, 225, 511, 512, 513, 895, 896, 897, 4095, 4096, 4097, 9000)


def _graph():
    """A hub of every length, joined to random vertices of 12,000 that a sparse
    random graph links among themselves."""
    rng = np.random.default_rng(41)
    n, hubs = 12000, len(LENGTHS)
    s, d = [], []
    for h, deg in enumerate(LENGTHS):
        nb = rng.choice(np.arange(hubs, n), size=deg, replace=False)
        s.append(np.full(deg, h))
        d.append(nb)
    a, b = rng.integers(hubs, n, 9000), rng.integers(hubs, n, 9000)
    keep = a != b
    pairs = np.unique(np.stack([np.minimum(a[keep], b[keep]), np.maximum(a[keep], b[keep])], 1), axis=0)
    s.append(pairs[:, 0])
    d.append(pairs[:, 1])
    colptr, rowidx = sg.csc_from_edges(n, np.concatenate(s).astype(np.int32), np.concatenate(d).astype(np.int32))
    assert tuple(sorted(np.diff(colptr)[:hubs])) == LENGTHS
    return n, colptr, rowidx


@pytest.mark.gpu
@pytest.mark.parametrize("hub_degree", [16, 600, 1 << 30])
@pytest.mark.parametrize("k,edges,colorings", [
    (3, U3, (1, 2, 3, 4, 5, 33)),  # rows of one value: up to 32 colorings a wavefront
    (5, U5, (1, 4, 5, 16)),    # rows of 4 and 6 values
    (6, STAR6, (3,)),
    (7, TREE7, (1, 3, 10)),    # rows of 6, 15 and 20 values
    (10, TREE10, (1, 4)),      # rows of 9 to 126 values: two wavefronts each
    (12, PATH12, (2,)),        # rows of up to 462 values: eight, a unit of all hubs at a time
])
def test_hub_lists_keep_the_reference_arithmetic(gpu_ctx, k, edges, colorings, hub_degree):
    """FP32 counts equal the oracle's restatement of the reference up to the
    order of the final FP64 sum over 12,000 vertices (12,000 * 2^-53 < 2e-12
    relative for a sum of non-negative terms); FP64 counts below 2^53 are
    equal, larger ones to the roundings of at most 9,000 + 12,000 additions
    (< 3e-12); and weighted FP64 counts to the same."""
    n, colptr, rowidx = _graph()
    keys = ("hub_degree", "exact_order")
    saved = [gpu_ctx.get_option(key) for key in keys]
    try:
        gpu_ctx.set_option("hub_degree", hub_degree)
        gpu_ctx.set_option("exact_order", 1)
        rng = np.random.default_rng(43 + k)
        weights = rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32)
        op = oracle.Plan(k, edges)
        for B in colorings:
            gpu_ctx.upload_graph(colptr, rowidx)
            plan = gpu_ctx.plan(k, edges)
            cols = rng.integers(0, k, size=(B, n)).astype(np.uint8)
            print(f"[hub] k={k} B={B}", flush=True)
            g32 = gpu_ctx.count(plan, B, colors=cols, precision="fp32")
            g64 = gpu_ctx.count(plan, B, colors=cols, precision="fp64")
            gpu_ctx.set_weights(weights)
            w64 = gpu_ctx.count(plan, B, colors=cols, precision="fp64")
            gpu_ctx.set_weights(None)
            for i in range(B):
                o32 = oracle.count_f32(op, colptr, rowidx, cols[i])
                o64 = oracle.count_f64(op, colptr, rowidx, cols[i])
                ow = oracle.count_f64(op, colptr, rowidx, cols[i], vals=weights)
                assert abs(g32[i] - o32) <= 2e-12 * abs(o32), (B, i, g32[i], o32)
                assert g64[i] == o64 if o64 < 2.0**53 else abs(g64[i] - o64) <= 3e-12 * o64, (B, i, g64[i], o64)
                assert abs(w64[i] - ow) <= 3e-12 * abs(ow), (B, i, w64[i], ow)
    finally:
        for key, v in zip(keys, saved):
            gpu_ctx.set_option(key, v)
