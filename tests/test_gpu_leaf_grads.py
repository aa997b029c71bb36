"""Entry gradients of one to six steps with a leaf aux child, up to four of them
in one launch (kept tables), against one launch per step (rebuilt tables)."""
import numpy as np
import pytest

import subgraph_amd as sg

KEYS = ("batch_tile", "adjoint_recompute")


def _star(k):
    return k, [(0, i) for i in range(1, k)]


TEMPLATES = {
    "path5": (5, [(0, 1), (1, 2), (2, 3), (3, 4)]),                          # one such step
    "star3": _star(3),
    "star4": _star(4),
    "star5": _star(5),                                                       # four
    "star7": _star(7),                                                       # four and two
    "tree7": (7, [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]),          # others between them
}


@pytest.mark.gpu
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("colorings,tile", [(1, 0), (4, 0), (5, 0), (7, 4)])
@pytest.mark.parametrize("name", sorted(TEMPLATES))
def test_steps_share_a_launch(gpu_ctx, name, colorings, tile, weighted):
    """Stars have no other step: the same tables and the same FP64 additions in
    the same order, so the same bits.  Else FP64 gradients at unit weights are
    integers (exact), with weights some thousand roundings apart at most."""
    k, edges = TEMPLATES[name]
    rng = np.random.default_rng(k + colorings)
    n = 300
    s, d = rng.integers(0, n, 1500), rng.integers(0, n, 1500)
    colptr, rowidx = sg.csc_from_edges(n, s[s != d].astype(np.int32), d[s != d].astype(np.int32))
    cols = rng.integers(0, k, size=(colorings, n)).astype(np.uint8)
    saved = [gpu_ctx.get_option(key) for key in KEYS]
    try:
        gpu_ctx.set_option("batch_tile", tile)
        gpu_ctx.upload_graph(colptr, rowidx)
        gpu_ctx.set_weights(rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32) if weighted else None)
        plan = gpu_ctx.plan(k, edges)
        for precision in ("fp64", "fp32"):
            got = []
            for rebuilt in (0, 1):
                gpu_ctx.set_option("adjoint_recompute", rebuilt)
                print(f"[leaf grads] {name} B={colorings} tile={tile} {precision} rebuilt={rebuilt}", flush=True)
                for _ in range(2):  # the second call replays the first's graph
                    raw, grad = gpu_ctx.count_grad(plan, colorings, colors=cols, precision=precision)
                got.append((raw, grad))
            (r0, g0), (r1, g1) = got
            assert np.array_equal(r0, r1)
            if name.startswith("star") or (precision == "fp64" and not weighted):
                assert np.array_equal(g0, g1)
            elif precision == "fp64":
                assert np.all(np.abs(g0 - g1) <= 1e-12 * np.abs(g1))
    finally:
        gpu_ctx.set_weights(None)
        for key, v in zip(KEYS, saved):
            gpu_ctx.set_option(key, v)
