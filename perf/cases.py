"""The work that the measurements of this library stand for: colorful counts
and their gradients through the package's public calls, from the smallest
one-coloring count to the largest forward+backward that one GPU holds.

A case is a graph (R-MAT with the usual quadrant probabilities, or uniformly
random edges; vertices without an edge removed, as the text loader removes
them), a template tree, a number of colorings and a precision:

  kind "count"  Context.count: the raw colorful count of each coloring
  kind "multi"  Context.count_multi: an uneven batch of three templates
  kind "train"  autograd.colorful_count with per-entry weights U(0.5, 1.5),
                and the gradient of a weighted sum of the counts
  kind "grad"   Context.count_grad_device at unit weights: the counts and, per
                entry, the number of colorful maps that use it

Everything a program keeps between calls (the uploaded graph, the plans, the
weight and gradient buffers) is made in prepare(); the graph's vertex numbers,
the weights, the colors and the color stream all come from the seed.
"""
import itertools

import numpy as np
import torch

import subgraph_amd as sg
from subgraph_amd.autograd import colorful_count

TEMPLATES = {
    "u3": (3, [(0, 1), (1, 2)]),
    "u5": (5, [(0, 1), (1, 2), (2, 3), (3, 4)]),
    "star5": (5, [(0, 1), (0, 2), (0, 3), (0, 4)]),
    "tree7": (7, [(0, 1), (1, 2), (2, 3), (1, 4), (4, 5), (4, 6)]),
    "tree10": (10, [(0, 1), (1, 2), (2, 3), (3, 4), (1, 5), (5, 6), (5, 7), (7, 8), (7, 9)]),
    "tree12": (12, [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5), (2, 6), (6, 7), (7, 8), (6, 9), (9, 10), (10, 11)]),
}
MIXED = (("u5", 16), ("tree7", 10), ("tree10", 4))


def _case(name, kind, template, graph, n, ef, colorings, precision="fp32", colors="stream", tile=0):
    c = {"kind": kind, "template": template, "graph": graph, "n": n, "ef": ef, "colorings": colorings,
         "precision": precision, "colors": colors, "tile": tile}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest use: one coloring of the 3-path on a small graph, where
        # a call is launches and host work
        _case("u3_s16_one", "count", "u3", "rmat", 1 << 16, 16, 1),
        # the reference's own method: one coloring per call, a mid-sized graph
        _case("tree7_s20_one", "count", "tree7", "rmat", 1 << 20, 8, 1),
        # an estimate: many colorings of that template in one call
        _case("tree7_s20_64", "count", "tree7", "rmat", 1 << 20, 8, 64),
        # a narrow template over a graph with large hubs, a usual batch
        _case("u5_s18_16", "count", "u5", "rmat", 1 << 18, 16, 16),
        # exact integer counts in FP64 tables, the caller's own colors
        _case("tree10_s18_fp64", "count", "tree10", "rmat", 1 << 18, 16, 4, "fp64", "caller"),
        # the widest template, counts only
        _case("tree12_s20_4", "count", "tree12", "rmat", 1 << 20, 16, 4, tile=4),
        # several templates in one call
        _case("mixed_s18", "multi", "mixed", "rmat", 1 << 18, 16, 30),
        # a training step on edge weights, one coloring
        _case("star5_s18_train_one", "train", "star5", "rmat", 1 << 18, 16, 1),
        # a training step of a batch of colorings
        _case("u5_s18_train_16", "train", "u5", "rmat", 1 << 18, 16, 16),
        # a graph without hubs and of no round size: per-entry counts in FP64
        _case("tree7_uniform_grad", "grad", "tree7", "uniform", 300007, 12, 5, "fp64"),
        # the headline's step (widest template, 4 colorings per pass) on a
        # graph of which several fit the card
        _case("tree12_s20_grad_4", "grad", "tree12", "rmat", 1 << 20, 16, 4, tile=4),
        # the largest graph, one coloring forward and backward
        _case("tree12_s22_grad_one", "grad", "tree12", "rmat", 1 << 22, 16, 1, tile=1),
    ]


# colorings of a drawn case at most, by template, for graphs of up to 2^20 n * ef / 2^24
_MOST = {"u3": 64, "u5": 64, "star5": 64, "tree7": 64, "tree10": 16, "tree12": 4}


def draw(rng):
    """One more case: any template, kind and precision over graphs of 2^14 to
    2^20 vertices (sizes spread over their logarithm, odd ones among them)."""
    n = int(round(2 ** rng.uniform(14, 20)))
    ef = rng.choice((4, 8, 11, 16))
    graph = rng.choice(("rmat", "rmat", "rmat", "uniform"))
    kind = rng.choice(("count", "count", "count", "multi", "train", "grad", "grad"))
    if kind == "multi":
        return _case(None, kind, "mixed", graph, min(n, 1 << 18), ef, 30)
    template = rng.choice(sorted(TEMPLATES))
    precision = rng.choice(("fp32", "fp32", "fp64"))
    most = _MOST[template]
    if precision == "fp64" or kind != "count":
        most = max(1, most // 4)
    b = min(most, int(round(2 ** rng.uniform(0, 6))))
    colors = rng.choice(("stream", "caller")) if kind == "count" else "stream"
    return _case(None, kind, template, graph, n, ef, b, precision, colors, tile=b if template == "tree12" else 0)


# ------------------------------------------------------------------ inputs

def _graph(case, seed):
    """The case's graph as CSC on the GPU (int64): (n, colptr, rowidx).  Its
    shape is the case's; the vertex numbers, and with them the entries' order,
    come from the seed."""
    g = torch.Generator("cuda").manual_seed(17)
    n0, m = case["n"], case["n"] * case["ef"]
    if case["graph"] == "rmat":
        src = torch.zeros(m, dtype=torch.int64, device="cuda")
        dst = torch.zeros(m, dtype=torch.int64, device="cuda")
        for _ in range((n0 - 1).bit_length()):
            r = torch.rand(m, generator=g, device="cuda")
            lower = r >= 0.76
            src = src * 2 + lower
            dst = dst * 2 + (((r >= 0.57) & ~lower) | (r >= 0.95))
    else:
        src = torch.randint(n0, (m,), generator=g, device="cuda")
        dst = torch.randint(n0, (m,), generator=g, device="cuda")
    keep = (src != dst) & (src < n0) & (dst < n0)
    src, dst = src[keep], dst[keep]
    key = torch.unique(torch.minimum(src, dst) * n0 + torch.maximum(src, dst))
    src, dst = key // n0, key % n0
    used = torch.zeros(n0, dtype=torch.int64, device="cuda")
    used[src] = 1
    used[dst] = 1
    place = torch.cumsum(used, 0) - 1
    n = int(used.sum())
    place = torch.randperm(n, generator=g.manual_seed(1000003 * seed + 17), device="cuda")[place]
    src, dst = place[src], place[dst]
    both = torch.sort(torch.cat([src * n + dst, dst * n + src])).values
    rows = both % n
    colptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    colptr[1:] = torch.cumsum(torch.bincount(both // n, minlength=n), 0)
    return n, colptr, rows


def _weights(nnz, seed):
    g = torch.Generator("cuda").manual_seed(1000003 * seed + 29)
    return torch.rand(nnz, generator=g, device="cuda") + 0.5


def _cotangent(case, seed):
    return np.random.RandomState(seed % 2**31).uniform(0.5, 1.5, case["colorings"])


def _stream(seed):
    return 7919 * seed + 101  # the device's color stream of this seed


def _caller_colors(case, n, k, seed):
    return np.random.RandomState(seed % 2**31).randint(0, k, (case["colorings"], n)).astype(np.uint8)


def prepare(case, seed):
    n, colptr, rows = _graph(case, seed)
    ctx = sg.Context(0)
    if case["tile"]:
        ctx.set_option("batch_tile", case["tile"])
    ctx.upload_graph(colptr.to(torch.int32).cpu().numpy(), rows.to(torch.int32).cpu().numpy())
    nnz = rows.numel()
    del colptr, rows
    s = {"case": case, "ctx": ctx, "seed": _stream(seed)}
    if case["kind"] == "multi":
        s["plans"] = [ctx.plan(*TEMPLATES[t]) for t, _ in MIXED]
        return s
    nv, edges = TEMPLATES[case["template"]]
    s["plan"] = ctx.plan(nv, edges)
    if case["kind"] == "count" and case["colors"] == "caller":
        s["colors"] = _caller_colors(case, n, nv, seed)
    elif case["kind"] == "train":
        s["weights"] = _weights(nnz, seed).requires_grad_()
        s["cotangent"] = torch.from_numpy(_cotangent(case, seed)).to("cuda")
    elif case["kind"] == "grad":
        dtype = torch.float32 if case["precision"] == "fp32" else torch.float64
        s["grad"] = torch.empty(nnz, dtype=dtype, device="cuda")
        s["cotangent"] = _cotangent(case, seed)
    torch.cuda.empty_cache()  # the graph's construction left blocks the library's tables may need
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    b, precision = case["colorings"], case["precision"]
    if case["kind"] == "count":
        if "colors" in s:
            return ctx.count(s["plan"], b, colors=s["colors"], precision=precision)
        return ctx.count(s["plan"], b, seed=s["seed"], precision=precision)
    if case["kind"] == "multi":
        return ctx.count_multi(s["plans"], [c for _, c in MIXED], [s["seed"] + i for i in range(len(MIXED))],
                               precision=precision)
    if case["kind"] == "train":
        raw = colorful_count(s["weights"], ctx, s["plan"], b, seed=s["seed"], precision=precision)
        grad, = torch.autograd.grad(raw, s["weights"], s["cotangent"])
        return raw.detach(), grad
    raw = ctx.count_grad_device(s["plan"], b, s["grad"].data_ptr(), seed=s["seed"], precision=precision,
                                cotangent=s["cotangent"])
    return raw, s["grad"]


# ------------------------------------------------------- work and the truth

def _steps(nv, edges):
    """The tree's dynamic program from template vertex 0: (size of the table
    so far, size of the child's table) of every join."""
    near = {v: [] for v in range(nv)}
    for a, b in edges:
        near[a].append(b)
        near[b].append(a)

    def size(v, parent):
        return 1 + sum(size(u, v) for u in near[v] if u != parent)

    out = []

    def walk(v, parent):
        a = 1
        for u in near[v]:
            if u != parent:
                walk(u, v)
                out.append((a, size(u, v)))
                a += out[-1][1]

    walk(0, -1)
    return out


def _choose(n, r):
    v = 1
    for i in range(r):
        v = v * (n - i) // (i + 1)
    return v


def _flops(template, n, nnz):
    """Additions and multiplications of one coloring forward: for each join,
    one addition per entry and set of the child's table that avoids the
    vertex's color, and two operations per split."""
    nv, edges = TEMPLATES[template]
    f = 0
    for a, b in _steps(nv, edges):
        f += nnz * _choose(nv - 1, b) * b / (nv - 1)
        f += 2 * n * _choose(nv - 1, a + b - 1) * _choose(a + b - 1, a - 1)
    return f


def work(case):
    n, nnz = case["n"], 2 * case["n"] * case["ef"]
    size = 8 if case["precision"] == "fp64" else 4
    moved = 4 * (n + 1) + 4 * nnz
    parts = MIXED if case["kind"] == "multi" else ((case["template"], case["colorings"]),)
    flops = sum(b * _flops(t, n, nnz) for t, b in parts)
    if case["colors"] == "caller":
        moved += case["colorings"] * n
    if case["kind"] in ("train", "grad"):
        flops *= 3  # forward, and for every product of it two in the adjoint
        moved += nnz * (8 if case["kind"] == "train" else size)
    return {"bytes": moved + 8 * case["colorings"], "flops": flops}


def _mix(x):
    """splitmix64's finalizer on int64 tensors (wrapping arithmetic)."""
    def shr(v, s):
        return (v >> s) & ((1 << (64 - s)) - 1)
    def wrap(v):
        return v - (1 << 64) if v >= 1 << 63 else v
    x = x + wrap(0x9E3779B97F4A7C15)
    x = (x ^ shr(x, 30)) * wrap(0xBF58476D1CE4E5B9)
    x = (x ^ shr(x, 27)) * wrap(0x94D049BB133111EB)
    return x ^ shr(x, 31)


def _stream_colors(seed, coloring, n, k):
    """Coloring `coloring` of the documented color stream."""
    gold = 0x9E3779B97F4A7C15 * coloring % (1 << 64)
    gold -= (1 << 64) if gold >= 1 << 63 else 0
    v = torch.arange(n, dtype=torch.int64, device="cuda") + gold
    h = _mix(_mix(v) ^ seed)
    return (((h >> 32) & 0xFFFFFFFF) * k) >> 32


def _matrix(n, rowptr, cols, w):
    return torch.sparse_csr_tensor(rowptr, cols, torch.ones_like(cols, dtype=torch.float64) if w is None else w, (n, n))


def _joins(k, a, b):
    """[sets of size a + b][splits]: the index of the part of size a and of
    the rest, over sets of k colors in lexicographic order."""
    place = [{c: i for i, c in enumerate(itertools.combinations(range(k), r))} for r in (a, b)]
    left, right = [], []
    for whole in itertools.combinations(range(k), a + b):
        parts = list(itertools.combinations(whole, a))
        left.append([place[0][p] for p in parts])
        right.append([place[1][tuple(c for c in whole if c not in p)] for p in parts])
    return torch.tensor(left, device="cuda").T, torch.tensor(right, device="cuda").T


def _truth(template, n, graph, w, colors, cotangent, grad):
    """The colorful count of one coloring in FP64 and, added to `grad`, its
    derivatives times `cotangent` (entries sorted by row)."""
    rowptr, owner, cols, back = graph
    nv, edges = TEMPLATES[template]
    near = {v: [] for v in range(nv)}
    for a, b in edges:
        near[a].append(b)
        near[b].append(a)
    tape = []
    matrix = _matrix(n, rowptr, cols, w)

    def walk(v, parent):
        t, a = torch.nn.functional.one_hot(colors, nv).double(), 1
        for u in near[v]:
            if u == parent:
                continue
            child, b = walk(u, v)
            left, right = _joins(nv, a, b)
            y = matrix @ child
            out = torch.zeros(n, left.shape[1], dtype=torch.float64, device="cuda")
            for i, j in zip(left, right):
                out.addcmul_(t[:, i], y[:, j])
            if grad is not None:
                tape.append((t, child, y, out, left, right))
            t, a = out, a + b
        return t, a

    root, _ = walk(0, -1)
    raw = float(root.sum())
    if grad is not None:
        # the transposed matrix: the weight of entry (v, u) moved to row u
        turned = matrix if w is None else _matrix(n, rowptr, cols, w[back])
        adjoint = {id(root): torch.full_like(root, cotangent)}
        for t, child, y, out, left, right in reversed(tape):
            g = adjoint.pop(id(out))
            dt, dy = torch.zeros_like(t), torch.zeros_like(y)
            for into, by, other, x in ((dt, left, right, y), (dy, right, left, t)):
                # every set has the same number of splits it is a part of
                order = torch.sort(by.T.reshape(-1), stable=True).indices.reshape(into.shape[1], -1).T
                for places in order:
                    into.addcmul_(g[:, places // len(left)], x[:, other.T.reshape(-1)[places]])
            step = max(1, (1 << 26) // y.shape[1])
            for e in range(0, cols.numel(), step):
                grad[e:e + step] += (dy[owner[e:e + step]] * child[cols[e:e + step]]).sum(1)
            adjoint[id(child)] = turned @ dy
            adjoint[id(t)] = dt
    return raw


def exact(case, seed):
    """run()'s values in FP64 by plain tensor operations; None where that
    takes too long or too much memory."""
    if case["template"] == "tree12" and (case["n"] > 1 << 20 or case["n"] * case["ef"] * case["colorings"] > 1 << 26):
        return None
    if case["n"] * case["ef"] * case["colorings"] > 1 << 28 and case["template"] in ("tree10", "tree12"):
        return None
    n, colptr, rows = _graph(case, seed)
    owner_col = torch.repeat_interleave(torch.arange(n, device="cuda"), colptr[1:] - colptr[:-1])
    # entry e is (row rows[e], column owner_col[e]); the pattern is symmetric
    # and the list sorted by column then row, so sorting by row then column
    # visits each entry's transpose in turn
    order = torch.argsort(rows * n + owner_col)
    cols = owner_col[order]
    graph = (colptr, owner_col, cols, order)
    parts = MIXED if case["kind"] == "multi" else ((case["template"], case["colorings"]),)
    w = None
    if case["kind"] == "train":
        w = _weights(rows.numel(), seed).double()[order]
    wants_grad = case["kind"] in ("train", "grad")
    cot = _cotangent(case, seed)
    grad = torch.zeros(rows.numel(), dtype=torch.float64, device="cuda") if wants_grad else None
    out = []
    for i, (template, b) in enumerate(parts):
        k = TEMPLATES[template][0]
        raw = np.zeros(b)
        for c in range(b):
            if case["kind"] == "count" and case["colors"] == "caller":
                colors = torch.from_numpy(_caller_colors(case, n, k, seed)[c]).to("cuda").long()
            else:
                colors = _stream_colors(_stream(seed) + i, c, n, k)
            raw[c] = _truth(template, n, graph, w, colors, float(cot[c]) if wants_grad else 0.0, grad)
        out.append(raw)
    if case["kind"] == "multi":
        return out
    if not wants_grad:
        return out[0]
    by_entry = torch.empty_like(grad)
    by_entry[order] = grad
    return (torch.from_numpy(out[0]), by_entry) if case["kind"] == "train" else (out[0], by_entry)
