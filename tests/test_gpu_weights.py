"""Entry weights across precisions: the FP64 copy is made by the first FP64
pass after the weights were set, so every order of sets, FP32 and FP64 passes,
counts, batches of templates and gradients has to see the current ones."""
import numpy as np
import pytest

import oracle
import subgraph_amd as sg

U5 = [(0, 1), (1, 2), (2, 3), (3, 4)]
STAR5 = [(0, 1), (0, 2), (0, 3), (0, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("edges", [U5, STAR5])
def test_current_weights_in_every_order_of_passes(gpu_ctx, edges):
    """FP64 counts equal the oracle's to 1e-12 (some 1e4 non-negative terms),
    FP32 ones to 1e-5 (the parity bar), and FP64 gradients satisfy
    sum_e w_e * grad_e = (k - 1) * count to 1e-12, after each change of the
    weights and whichever precision ran before."""
    rng = np.random.default_rng(7)
    n = 300
    a, b = rng.integers(0, n, 2500), rng.integers(0, n, 2500)
    pairs = np.unique(np.stack([np.minimum(a, b), np.maximum(a, b)], 1)[a != b], axis=0)
    colptr, rowidx = sg.csc_from_edges(n, pairs[:, 0].copy(), pairs[:, 1].copy())
    gpu_ctx.upload_graph(colptr, rowidx)
    plan, op = gpu_ctx.plan(5, edges), oracle.Plan(5, edges)
    cols = rng.integers(0, 5, size=(2, n)).astype(np.uint8)
    seeds = [3, 4]
    try:
        for order in ("fp32 fp64 grad", "fp64 fp32 grad", "grad fp64 fp32", "multi fp32 fp64"):
            w = rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32)
            gpu_ctx.set_weights(w)
            want = np.array([oracle.count_f64(op, colptr, rowidx, c, vals=w) for c in cols])
            for what in order.split():
                print(f"[weights] {order}: {what}", flush=True)
                if what == "grad":
                    raw, grad = gpu_ctx.count_grad(plan, 2, colors=cols, precision="fp64")
                    assert np.allclose(raw, want, rtol=1e-12, atol=0)
                    assert abs((grad * w).sum() - 4 * want.sum()) <= 1e-12 * 4 * want.sum()
                elif what == "multi":
                    got = gpu_ctx.count_multi([plan, plan], [1, 1], seeds, precision="fp64")
                    for g, s in zip(got, seeds):
                        o = oracle.count_f64(op, colptr, rowidx, sg.colors_fill(s, 0, 1, n, 5)[0], vals=w)
                        assert abs(g[0] - o) <= 1e-12 * o
                else:
                    got = gpu_ctx.count(plan, 2, colors=cols, precision=what)
                    assert np.allclose(got, want, rtol=1e-12 if what == "fp64" else 1e-5, atol=0)
    finally:
        gpu_ctx.set_weights(None)
