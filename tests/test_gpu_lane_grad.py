"""The transposed gather that also takes the entries' gradients (one gather per
step) against the separate gradient and transposed gathers (fuse_grad 0), over
the templates, batch sizes and passes in which its shape changes."""
import numpy as np
import pytest

import subgraph_amd as sg

TEMPLATES = {
    "u3": (3, [(0, 1), (1, 2)]),
    "u5": (5, [(0, 1), (1, 2), (2, 3), (3, 4)]),
    "tree7": (7, [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]),
    "tree10": (10, [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]),
    "tree12": (12, [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (2, 6), (6, 7), (7, 8), (6, 9), (9, 10), (10, 11)]),
}
KEYS = ("fuse_grad", "hub_degree", "hub_chunk", "batch_tile", "adjoint_recompute")


@pytest.mark.gpu
@pytest.mark.parametrize("name,colorings,tile", [
    ("u3", 1, 0), ("u3", 64, 0), ("u5", 1, 0), ("u5", 5, 2), ("u5", 16, 0), ("tree7", 1, 0), ("tree7", 5, 3),
    ("tree7", 11, 0), ("tree10", 2, 0), ("tree12", 1, 0), ("tree12", 3, 2),
])
@pytest.mark.parametrize("hub_degree,hub_chunk", [(512, 1024), (16, 24)])
def test_one_gather_gives_the_gradients_of_two(gpu_ctx, name, colorings, tile, hub_degree, hub_chunk):
    """At unit weights FP64 counts and gradients are sums of integers: equal
    where every partial sum stays below 2^53, else to some thousand roundings
    of a non-negative sum (1e-11 in norm).  With weights U(0.5, 1.5) the same;
    FP32 gradients agree in norm to 1e-5, and the identity sum_e w_e grad_e =
    (k - 1) * count holds in FP64 to 1e-11, also with rebuilt tables."""
    k, edges = TEMPLATES[name]
    saved = [gpu_ctx.get_option(key) for key in KEYS]
    rng = np.random.default_rng(k + colorings)
    src, dst = sg.rmat_edges(9, 6, seed=3)
    n = 1 << 9
    colptr, rowidx = sg.csc_from_edges(n, src, dst)
    w = rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32)
    cols = rng.integers(0, k, size=(colorings, n)).astype(np.uint8)
    cot = rng.integers(1, 4, colorings).astype(np.float64)
    try:
        gpu_ctx.set_option("hub_degree", hub_degree)
        gpu_ctx.set_option("hub_chunk", hub_chunk)
        gpu_ctx.set_option("batch_tile", tile)
        gpu_ctx.upload_graph(colptr, rowidx)
        plan = gpu_ctx.plan(k, edges)
        for weights in (None, w):
            gpu_ctx.set_weights(weights)
            got = {}
            for fuse, rec in ((1, 0), (0, 0), (1, 1)):
                gpu_ctx.set_option("fuse_grad", fuse)
                gpu_ctx.set_option("adjoint_recompute", rec)
                for precision in ("fp64", "fp32"):
                    print(f"[lane grad] {name} B={colorings} tile={tile} hub={hub_degree} fuse={fuse} rec={rec} "
                          f"{precision} weighted={weights is not None}", flush=True)
                    got[fuse, rec, precision] = gpu_ctx.count_grad(plan, colorings, colors=cols, precision=precision,
                                                                   cotangent=cot)
            raw, grad = got[0, 0, "fp64"]
            scale = np.linalg.norm(grad)
            exact = weights is None and grad.max() < 2.0**53
            for key, (r, g) in got.items():
                if key[2] == "fp64":
                    assert np.array_equal(r, raw) or np.allclose(r, raw, rtol=1e-12, atol=0), key
                    if exact:
                        assert np.array_equal(g, grad), key
                    assert np.linalg.norm(g - grad) <= 1e-11 * scale, key
                    ww = np.ones(len(rowidx)) if weights is None else w.astype(np.float64)
                    total = (k - 1) * (cot * r).sum()
                    assert abs((g * ww).sum() - total) <= 1e-11 * abs(total), key
                else:
                    assert np.allclose(r, raw, rtol=1e-5, atol=0), key
                    assert np.linalg.norm(g - grad) <= 1e-5 * scale, key
    finally:
        gpu_ctx.set_weights(None)
        for key, v in zip(KEYS, saved):
            gpu_ctx.set_option(key, v)
