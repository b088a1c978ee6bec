"""The work that a user of this framework has it do, as measurable cases.

Three public calls make up the path: a reordering (``sporder.chunk_similarity_greedy``,
or ``sporder.chunk_greedy`` on the global sketch), the permutation apply
(``sporder.reorder``) and the CSR SpMM they feed (``sporder.spmm_csr``, its
planned form, and the scaled operator of the GCN example).  A case is one call,
or the three in a row, on a seeded sparse matrix made on the GPU:

  planted  hidden 64-column blocks, 80 % of a row's nonzeros inside its block;
           rows scrambled (as the benchmark's configurations) or kept in block
           order; not symmetric
  grid     7-point stencil in natural order, 2 % of the couplings missing
  fem      27-point stencil with 3 unknowns per node (an elasticity matrix of
           about 80 nonzeros per row), 2 % of the couplings missing
  rgg      random geometric graph, points numbered cell by cell
  power    Chung-Lu graph of exponent 2.1 with self loops, ids scrambled
"""

import math

import torch

from chunkedgreedy_amd import e2e_gcn, sporder

DEVICE = "cuda:0"


def listed():
    return [
        # A small graph reordered on the fly (the sizes of citation graphs and
        # of the repository's own plumbing configuration): latency.
        {"name": "csg_small", "op": "csg", "matrix": "planted", "n": 20_000, "deg": 10},
        # A mesh-like graph of the size of rgg_n_2_20: an ordinary reordering.
        {"name": "csg_rgg", "op": "csg", "matrix": "rgg", "n": 1 << 20, "deg": 13},
        # A finite-element matrix: long rows with close neighbours, k past 64.
        {"name": "csg_fem", "op": "csg", "matrix": "fem", "g": 40},
        # A social-network graph of the size of ogbn-products: hubs.
        {"name": "csg_power", "op": "csg", "matrix": "power", "n": 2_449_029, "deg": 25},
        # The global-sketch reordering on a mid-size mesh.
        {"name": "cg_rgg", "op": "cg", "matrix": "rgg", "n": 1 << 18, "deg": 13},
        # The benchmark's step: reorder, apply, SpMM at N = 128.
        {"name": "step_planted", "op": "step", "matrix": "planted", "n": 1 << 20, "deg": 16,
         "N": 128},
        # P A P^T with values, from a reordering of the same matrix.
        {"name": "apply_rgg", "op": "apply", "matrix": "rgg", "n": 1 << 20, "deg": 13,
         "symmetric": True},
        # One SpMM on a small graph: latency and launches.
        {"name": "spmm_small_32", "op": "spmm", "matrix": "planted", "n": 20_000, "deg": 10,
         "N": 32, "plan": False},
        # Multi-vector product of a stencil solver, planned once and reused.
        {"name": "spmm_grid_64", "op": "spmm", "matrix": "grid", "g": 160, "N": 64,
         "plan": True},
        # A graph layer whose width is its number of classes (47): odd width, hubs.
        {"name": "spmm_power_47", "op": "spmm", "matrix": "power", "n": 300_000, "deg": 25,
         "N": 47, "plan": True},
        # Rows that share columns: the blocked plan.
        {"name": "spmm_fem_128", "op": "spmm", "matrix": "fem", "g": 40, "N": 128,
         "plan": True},
        # The GCN's normalised operator, forward and backward, at its hidden width.
        {"name": "gcn_power_128", "op": "gcn", "matrix": "power", "n": 2_449_029, "deg": 25,
         "N": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["csg"] * 5 + ["spmm"] * 4 + ["apply"] * 2 + ["step"] * 2 + ["cg", "gcn"])
    if op == "cg":
        kinds = ["rgg", "grid", "planted"]
    elif op == "gcn":
        kinds = ["power", "rgg"]
    else:
        kinds = ["planted", "grid", "fem", "rgg", "power"]
    kind = rng.choice(kinds)
    small = op == "cg"
    case = {"op": op, "matrix": kind}
    if kind == "grid":
        case["g"] = _log(rng, 12, 60 if small else 120)
    elif kind == "fem":
        case["g"] = _log(rng, 8, 36)
    else:
        lo = 20_000 if kind == "power" else 2_000
        case["n"] = _log(rng, lo, 150_000 if small else 900_000)
        case["deg"] = rng.randint(6, 14 if small else 25)
        if kind == "planted":
            case["keep"] = rng.random() < 0.5
    if op in ("csg", "cg") and rng.random() < 0.5:
        case["k"] = rng.choice([16, 16, 24, 32])
        case["oversampling"] = rng.choice([2.0, 4.0, 8.0])
    if op == "csg":
        case["chunk_size"] = rng.choice([0, 0, 0, 256, 500, 2048])
        case["stats"] = rng.random() < 0.2
    if op in ("spmm", "step", "gcn"):
        case["N"] = rng.choice([8, 16, 32, 64, 96, 100, 128, 256, rng.randint(1, 150)])
    if op == "spmm":
        case["plan"] = rng.random() < 0.7
    if op == "apply":
        case["symmetric"] = rng.random() < 0.7
    return case


# ---- the matrices -------------------------------------------------------------


def _csr(n, rows, cols):
    """(ptr, ind) int32 of distinct (row, col) pairs."""
    keys = torch.sort(rows * n + cols).values
    counts = torch.bincount(keys // n, minlength=n)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(counts, 0, out=ptr[1:])
    return ptr.to(torch.int32), (keys % n).to(torch.int32)


def _mirrored(n, a, b, diagonal=True):
    """The symmetric pattern of the distinct pairs a != b, with the diagonal or without."""
    i = torch.arange(n if diagonal else 0, device=DEVICE)
    return _csr(n, torch.cat([i, a, b]), torch.cat([i, b, a]))


def _some(count, keep, gen):
    """`keep` of range(count), at random."""
    return torch.randperm(count, generator=gen, device=DEVICE)[:keep]


def _planted(n, deg, keep, gen):
    width = 64
    n_in = max(1, round(0.8 * deg))
    n_out = deg - n_in
    pick = torch.rand((n, width), generator=gen, device=DEVICE).topk(n_in, 1).indices
    start = torch.arange(n, device=DEVICE).div(width, rounding_mode="floor") * width
    start = start.clamp_(max=n - width)[:, None]
    cols = [start + pick]
    if n_out:
        # One column from each of n_out equal parts of the columns outside the block.
        u = torch.rand((n, n_out), generator=gen, device=DEVICE, dtype=torch.float64)
        part = (n - width) // n_out
        cols.append((start + width + torch.arange(n_out, device=DEVICE) * part
                     + (u * part).long()) % n)
    cols = torch.randperm(n, generator=gen, device=DEVICE)[torch.cat(cols, 1)]
    rows = torch.arange(n, device=DEVICE)
    if not keep:
        rows = torch.randperm(n, generator=gen, device=DEVICE)
    return _csr(n, rows[:, None].expand_as(cols).reshape(-1), cols.reshape(-1))


def _couplings(g, offsets, gen):
    """Node pairs (a, b) of a g^3 grid for the given offsets, 2 % missing."""
    i = torch.arange(g ** 3, device=DEVICE)
    x, y, z = i % g, i.div(g, rounding_mode="floor") % g, i.div(g * g, rounding_mode="floor")
    a, b = [], []
    for dx, dy, dz in offsets:
        ok = (x + dx >= 0) & (x + dx < g) & (y + dy >= 0) & (y + dy < g) & (z + dz < g)
        at = ok.nonzero()[:, 0]
        at = at[_some(at.numel(), at.numel() - at.numel() // 50, gen)]
        a.append(at)
        b.append(at + dx + g * dy + g * g * dz)
    return torch.cat(a), torch.cat(b)


_GRID = [(1, 0, 0), (0, 1, 0), (0, 0, 1)]
_FEM = [(x, y, z) for z in (0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)
        if (z, y, x) > (0, 0, 0)]


def _couplings_count(g, offsets):
    counts = [(g - abs(x)) * (g - abs(y)) * (g - z) for x, y, z in offsets]
    return sum(c - c // 50 for c in counts)


def _grid(g, gen):
    return _mirrored(g ** 3, *_couplings(g, _GRID, gen))


def _fem(g, gen):
    a, b = _couplings(g, _FEM, gen)
    i = torch.arange(g ** 3, device=DEVICE)
    r, c = torch.cat([i, a, b]), torch.cat([i, b, a])
    d = torch.arange(3, device=DEVICE)
    rows = (3 * r[:, None, None] + d[None, :, None]).expand(-1, 3, 3)
    cols = (3 * c[:, None, None] + d[None, None, :]).expand(-1, 3, 3)
    return _csr(3 * g ** 3, rows.reshape(-1), cols.reshape(-1))


def _rgg(n, deg, gen):
    """The n * deg / 2 shortest of the pairs closer than 1.2 times the radius
    that gives about that many."""
    r = 1.2 * math.sqrt(deg / (math.pi * n))
    g = max(1, int(1 / r))
    pts = torch.rand((n, 2), generator=gen, device=DEVICE, dtype=torch.float64)
    cell = (pts * g).long().clamp_(max=g - 1)
    cid, order = torch.sort(cell[:, 1] * g + cell[:, 0], stable=True)
    pts, cell = pts[order], cell[order]
    start = torch.searchsorted(cid, torch.arange(g * g + 1, device=DEVICE))
    rows, cols, far = [], [], []
    for dx, dy in ((0, 0), (1, 0), (-1, 1), (0, 1), (1, 1)):
        ox, oy = cell[:, 0] + dx, cell[:, 1] + dy
        src = ((ox >= 0) & (ox < g) & (oy < g)).nonzero()[:, 0]
        nb = oy[src] * g + ox[src]
        cnt = start[nb + 1] - start[nb]
        a = torch.repeat_interleave(src, cnt)
        first = torch.cumsum(cnt, 0) - cnt
        b = torch.arange(a.numel(), device=DEVICE) + torch.repeat_interleave(
            start[nb] - first, cnt)
        d2 = (pts[a] - pts[b]).square().sum(1)
        near = (d2 < r * r) & (a < b)
        rows.append(a[near])
        cols.append(b[near])
        far.append(d2[near])
    at = torch.sort(torch.cat(far), stable=True).indices[: n * deg // 2]
    return _mirrored(n, torch.cat(rows)[at], torch.cat(cols)[at], diagonal=False)


def _power(n, deg, gen):
    w = (torch.arange(n, device=DEVICE, dtype=torch.float64) + 1) ** (-1 / 1.1)
    cum = torch.cumsum(w, 0)
    m = int(1.2 * n * deg)  # the hubs draw many edges twice: more than n * deg / 2 are left
    u, v = (torch.searchsorted(cum, torch.rand(m, generator=gen, device=DEVICE,
                                               dtype=torch.float64) * cum[-1]).clamp_(max=n - 1)
            for _ in range(2))
    a, b = torch.minimum(u, v), torch.maximum(u, v)
    edges = torch.unique((a * n + b)[a != b])
    edges = edges[_some(edges.numel(), n * deg // 2, gen)]
    p = torch.randperm(n, generator=gen, device=DEVICE)
    return _mirrored(n, p[edges // n], p[edges % n])


def _matrix(case, gen):
    kind = case["matrix"]
    if kind == "planted":
        return _planted(case["n"], case["deg"], case.get("keep", False), gen)
    if kind == "grid":
        return _grid(case["g"], gen)
    if kind == "fem":
        return _fem(case["g"], gen)
    if kind == "rgg":
        return _rgg(case["n"], case["deg"], gen)
    return _power(case["n"], case["deg"], gen)


def _sizes(case):
    """(n, nnz)."""
    kind = case["matrix"]
    if kind == "grid":
        g = case["g"]
        return g ** 3, g ** 3 + 2 * _couplings_count(g, _GRID)
    if kind == "fem":
        g = case["g"]
        return 3 * g ** 3, 9 * (g ** 3 + 2 * _couplings_count(g, _FEM))
    n, deg = case["n"], case["deg"]
    if kind == "planted":
        return n, n * deg
    return n, 2 * (n * deg // 2) + (n if kind == "power" else 0)


# ---- the cases ----------------------------------------------------------------


def _csg_options(case):
    return {"is_symmetric": case["matrix"] != "planted", "k": case.get("k", 0),
            "oversampling": case.get("oversampling", 0.0),
            "chunk_size": case.get("chunk_size", 0)}


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    ptr, ind = _matrix(case, gen)
    n, nnz = ptr.numel() - 1, ind.numel()
    op = case["op"]
    s = {"case": case, "ptr": ptr, "ind": ind}
    if op in ("csg", "cg"):
        s["options"] = _csg_options(case)
        if op == "csg":
            s["options"]["with_stats"] = case.get("stats", False)
        else:
            del s["options"]["chunk_size"]
        return s
    s["val"] = torch.rand(nnz, generator=gen, device=DEVICE) * 2 - 1
    if op == "apply":
        s["order"] = sporder.chunk_similarity_greedy(
            ptr, ind, is_symmetric=case["matrix"] != "planted")
        return s
    N = case["N"]
    s["B"] = torch.randn((n, N), generator=gen, device=DEVICE)
    if op == "spmm":
        s["plan"] = sporder.spmm_plan(ptr, ind) if case["plan"] else None
        s["out"] = torch.empty((n, N), device=DEVICE)
    elif op == "step":
        s["options"] = _csg_options(case)
        s["out"] = torch.empty((n, N), device=DEVICE)
    else:
        s["operator"] = e2e_gcn.GraphOp(ptr, ind, fused=True)
        s["grad"] = torch.randn((n, N), generator=gen, device=DEVICE)
    return s


def run(state):
    op, ptr, ind = state["case"]["op"], state["ptr"], state["ind"]
    if op == "csg":
        return sporder.chunk_similarity_greedy(ptr, ind, **state["options"])
    if op == "cg":
        return sporder.chunk_greedy(ptr, ind, **state["options"])
    if op == "apply":
        return sporder.reorder(ptr, ind, state["order"], val=state["val"],
                               symmetric=state["case"]["symmetric"])
    if op == "spmm":
        return sporder.spmm_csr(ptr, ind, state["val"], state["B"], out=state["out"],
                                plan=state["plan"])[0]
    if op == "step":
        order = sporder.chunk_similarity_greedy(ptr, ind, **state["options"])
        p2, i2, v2 = sporder.reorder(ptr, ind, order, val=state["val"], symmetric=True)
        C, _ = sporder.spmm_csr(p2, i2, v2, state["B"], out=state["out"])
        return {"order": order, "ptr": p2, "ind": i2, "val": v2, "C": C}
    # The operator is its own transpose: the backward pass applies it to the
    # gradient of its result.
    return {"y": state["operator"](state["B"]), "dx": state["operator"](state["grad"])}


def work(case):
    n, nnz = _sizes(case)
    op, N = case["op"], case.get("N", 0)
    pattern = 4 * (n + 1) + 4 * nnz
    order = pattern + 4 * n
    apply = 2 * pattern + 4 * n + 8 * nnz
    spmm = pattern + 4 * nnz + 8 * n * N
    if op in ("csg", "cg"):
        return {"bytes": order, "flops": 0}
    if op == "apply":
        return {"bytes": apply, "flops": 0}
    if op == "spmm":
        return {"bytes": spmm, "flops": 2 * nnz * N}
    if op == "step":
        return {"bytes": order + apply + spmm, "flops": 2 * nnz * N}
    # values and column scales per nonzero, a scale per row
    return {"bytes": 2 * (spmm + 4 * nnz + 4 * n), "flops": 2 * (3 * nnz * N + n * N)}


def tolerance(case):
    if case["op"] in ("csg", "cg"):
        # Orders are whole numbers; the statistics' means are 64-bit sums.
        return {"rel": 1e-9} if case.get("stats") else "exact"
    if case["op"] == "apply":
        return "exact"
    # 32-bit sums: the path is up to 2.7e-7 (2-norm) from the same sums in 64
    # bits where hub rows have chains of 512 terms, 1e-7 without them.
    return {"rel": 1e-6}


def _product64(ptr, ind, val, B):
    """A @ B in float64, by torch's own sparse product."""
    n = ptr.numel() - 1
    A = torch.sparse_csr_tensor(ptr.long(), ind.long(), val.double(), size=(n, n), device=DEVICE)
    return A @ B.double()


def exact(case, seed):
    op = case["op"]
    if op not in ("spmm", "gcn"):
        return None  # whole numbers, copied values, or a product that follows from them
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    ptr, ind = _matrix(case, gen)
    n, nnz = ptr.numel() - 1, ind.numel()
    val = torch.rand(nnz, generator=gen, device=DEVICE) * 2 - 1
    B = torch.randn((n, case["N"]), generator=gen, device=DEVICE)
    if op == "spmm":
        return _product64(ptr, ind, val, B)
    grad = torch.randn((n, case["N"]), generator=gen, device=DEVICE)
    d = (ptr[1:] - ptr[:-1]).double().clamp_min(1).rsqrt()
    one = torch.ones_like(val)
    return {"y": d[:, None] * _product64(ptr, ind, one, d[:, None] * B.double()),
            "dx": d[:, None] * _product64(ptr, ind, one, d[:, None] * grad.double())}
