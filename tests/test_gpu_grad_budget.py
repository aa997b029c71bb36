"""Gradients under memory budgets that hold the kept tables but not the Y rows
that the gathers with gradients need beside them."""
import numpy as np
import pytest

import subgraph_amd as sg

TREE7 = [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]
TREE10 = [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]
TREE12 = [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (2, 6), (6, 7), (7, 8), (6, 9), (9, 10), (10, 11)]
KEYS = ("fuse_grad", "adjoint_recompute", "mem_budget_mb")


@pytest.mark.gpu
@pytest.mark.parametrize("k,edges,scale,precision", [
    (7, TREE7, 15, "fp32"), (7, TREE7, 15, "fp64"), (10, TREE10, 15, "fp64"), (12, TREE12, 13, "fp32")])
def test_tables_that_just_fit_are_enough(gpu_ctx, k, edges, scale, precision):
    """The least budget of the separate gathers (fuse_grad 0, kept tables) is
    enough with fuse_grad 1, which then takes them for the steps whose node launch
    reads Y, all or the narrow ones (a step with a leaf main child reads none and keeps its one gather).
    FP64 gradients at unit weights are whole numbers: equal in any order below
    2^53, else to some thousand roundings (1e-11 in norm); FP32 ones to 1e-5 in
    norm.  Each budget's calls repeat their own bits, also beside passes of the
    same width under the other (another plan of the same captured shape)."""
    n = 1 << scale
    colptr, rowidx = sg.csc_from_edges(n, *sg.rmat_edges(scale, 8, seed=3))
    saved = [gpu_ctx.get_option(key) for key in KEYS]
    try:
        gpu_ctx.upload_graph(colptr, rowidx)
        plan = gpu_ctx.plan(k, edges)
        gpu_ctx.set_option("adjoint_recompute", 0)

        def grad(fuse, budget):
            gpu_ctx.set_option("fuse_grad", fuse)
            gpu_ctx.set_option("mem_budget_mb", budget)
            print(f"[budget] k={k} {precision} fuse={fuse} {budget} MB", flush=True)
            return gpu_ctx.count_grad(plan, 1, seed=9, precision=precision)

        least = 1
        while True:
            try:
                want = grad(0, least)
                break
            except sg.PGError:
                least += 1
                assert least < 1024
        first = {budget: grad(1, budget) for budget in (0, least, least * 11 // 10, least * 12 // 10)}
        exact = precision == "fp64" and want[1].max() < 2.0**53
        for raw, g in first.values():
            assert np.array_equal(raw, want[0])
            if exact:
                assert np.array_equal(g, want[1])
            assert np.linalg.norm(g - want[1]) <= (1e-5 if precision == "fp32" else 1e-11) * np.linalg.norm(want[1])
        for budget, (raw, g) in list(first.items()) * 2:
            again = grad(1, budget)
            assert np.array_equal(again[0], raw) and np.array_equal(again[1], g)
    finally:
        for key, v in zip(KEYS, saved):
            gpu_ctx.set_option(key, v)


@pytest.mark.gpu
def test_entry_buffers_are_left_room(gpu_ctx):
    """With little memory free, the tables of a gradient call leave room for its
    buffers per entry (some 28 bytes each beside the tables, of 1.3 GB free for
    18 million entries): the call runs, and gives what it gives with memory to
    spare, to FP32 rounding (1e-5, gradients in norm; a weighted histogram's order
    depends on the colorings of a pass)."""
    torch = pytest.importorskip("torch")
    n, mb = 150_000, 1 << 20
    rng = np.random.default_rng(103)
    a, b = rng.integers(0, n, 9_000_000), rng.integers(0, n, 9_000_000)
    key = np.unique(np.minimum(a, b)[a != b] * n + np.maximum(a, b)[a != b])
    colptr, rowidx = sg.csc_from_edges(n, (key // n).astype(np.int32), (key % n).astype(np.int32))
    ctx = sg.Context(0)
    ctx.upload_graph(colptr, rowidx)
    ctx.set_weights(rng.uniform(0.5, 1.5, len(rowidx)).astype(np.float32))
    plan = ctx.plan(7, TREE7)
    hold = []
    try:
        ctx.count(plan, 1, seed=9, precision="fp32")
        for keep, piece in ((4096, 2048), (1500, 128)):  # MB free, MB at a time
            while torch.cuda.mem_get_info()[0] > (keep + piece) * mb:
                hold.append(torch.empty(piece * mb, dtype=torch.uint8, device="cuda"))
        print(f"[tight memory] {torch.cuda.mem_get_info()[0] // mb} MB free, {len(rowidx)} entries", flush=True)
        raw, grad = ctx.count_grad(plan, 64, seed=9, precision="fp32")
        print(f"[tight memory] {ctx.get_option('last_tile')} colorings a pass", flush=True)
        assert 1 <= ctx.get_option("last_tile") < 64 and ctx.get_option("last_recompute") == 0
    finally:
        hold.clear()
        torch.cuda.empty_cache()
    ample, want = ctx.count_grad(plan, 64, seed=9, precision="fp32")
    assert ctx.get_option("last_tile") == 64
    assert np.allclose(raw, ample, rtol=1e-5, atol=0)
    assert np.linalg.norm(grad - want) <= 1e-5 * np.linalg.norm(want)
