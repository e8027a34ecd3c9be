"""Performance cases of the SpGEMM library: what its users run, through its public entry points.

Kinds of call
    product   one sparse product of device operands that are new to the context: set_operands, plan,
              symbolic, numeric (the two-phase device API, C in torch tensors)
    noalloc   the entry point that allocates nothing (dbd_spgemm_noalloc), C in arrays the caller keeps
    grad      forward and backward through spgemm_values (torch.autograd), loss 0.5 * sum(C * C)
    batch     one replay of a prepared batch of independent products (BatchRunner)
    host      host operands in, C in pinned host memory (Context.run in its d2h mode)

Matrices come from the library's seeded generators:
    er      uniform columns, a fixed number per row (A rows x inner, B inner x cols)
    mesh    columns near the diagonal, as of a mesh or a stencil: many products per entry of C
    web     web-like graph: short rows with a heavy tail, 70 % of the links near the row
    rmat    power-law graph (R-MAT .57/.19/.19), C = A * A; with `step` > 1, rows 0, step, 2 step, ..
            of it times the whole (odd steps: an R-MAT graph's even rows are its heavier ones)
    skewed  rows whose lengths follow a Zipf law (1.8), C = A * B
"""
import ctypes
import functools
import math
import random

import numpy as np
import torch

import dbd_amd
from dbd_amd._lib import check
from dbd_amd.autograd import spgemm_values
from dbd_amd.batch import BatchRunner, concat

#: Products of one drawn case at most (the largest listed ones have 5e8 and more).
MOST_PRODUCTS = 4.0e8


def listed():
    return [
        # a small system matrix squared: latency of the whole call
        {"name": "small_er_f64", "kind": "product", "gen": "er", "rows": 1000, "inner": 1000, "cols": 1000, "deg_a": 8,
         "deg_b": 8, "dtype": "f64", "block_rows": 4096},
        # a serving loop that may not allocate: one member-sized product, rows of uneven length
        {"name": "noalloc_skewed_f32", "kind": "noalloc", "gen": "skewed", "rows": 6007, "deg": 12.0, "dtype": "f32"},
        # Galerkin-like product of a mesh matrix: the same columns over and over (5 products an entry of C)
        {"name": "mesh_f64", "kind": "product", "gen": "mesh", "rows": 150000, "deg_min": 16, "deg_max": 56, "band": 64,
         "dtype": "f64", "block_rows": 4096},
        # circuit- and road-like matrix: a million very short rows
        {"name": "short_rows_f32", "kind": "product", "gen": "mesh", "rows": 1200007, "deg_min": 2, "deg_max": 7,
         "band": 12, "dtype": "f32", "block_rows": 4096},
        # two hops over a web graph of the size of the library's web benchmark
        {"name": "web_f64", "kind": "product", "gen": "web", "rows": 281903, "zipf": 2.1, "dtype": "f64",
         "block_rows": 4096},
        # the same graph with heavier rows, from host memory to host memory
        {"name": "web_host_f64", "kind": "host", "gen": "web", "rows": 281903, "zipf": 1.66, "dtype": "f64",
         "block_rows": 4096},
        # the library's benchmark: Erdos-Renyi 2,000,000 x 16 per row
        {"name": "er2m_f64", "kind": "product", "gen": "er", "rows": 2000000, "inner": 2000000, "cols": 2000000,
         "deg_a": 16, "deg_b": 16, "dtype": "f64", "block_rows": 512},
        # rectangular operands of odd sizes
        {"name": "rect_er_f32", "kind": "product", "gen": "er", "rows": 300007, "inner": 1000003, "cols": 777777,
         "deg_a": 9, "deg_b": 33, "dtype": "f32", "block_rows": 512},
        # friends of friends in a social graph: all row lengths up to hubs
        {"name": "rmat16_f64", "kind": "product", "gen": "rmat", "scale": 16, "edge": 16, "step": 1, "dtype": "f64",
         "block_rows": 512},
        # a sample of the rows of a large graph against all of it: long rows over many columns
        {"name": "rmat20_rows_f64", "kind": "product", "gen": "rmat", "scale": 20, "edge": 16, "step": 31,
         "dtype": "f64", "block_rows": 512},
        # training through the product: adjacency (normalised, self loops) times a learned sparse matrix
        {"name": "grad_rmat16_f32", "kind": "grad", "gen": "rmat", "scale": 16, "edge": 16, "step": 1, "dtype": "f32",
         "block_rows": 512},
        # many independent products in one replay
        {"name": "batch32_f32", "kind": "batch", "gen": "skewed", "members": 32, "rows_min": 1000, "rows_max": 60000,
         "deg_min": 4, "deg_max": 48, "dtype": "f32", "block_rows": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a family of matrices, a size spread over the logarithm of its range, a call."""
    gen = rng.choice(["er", "er", "mesh", "mesh", "web", "rmat", "rows", "skewed", "batch", "grad"])
    dtype = rng.choice(["f64", "f32"])
    block_rows = rng.choice([512, 4096])
    if gen == "batch":
        return {"kind": "batch", "gen": "skewed", "members": rng.randint(4, 40), "rows_min": 1000,
                "rows_max": _log(rng, 4000, 50000), "deg_min": 4, "deg_max": rng.randint(8, 48), "dtype": "f32",
                "block_rows": 4096}
    if gen == "grad":
        if rng.random() < 0.5:
            return {"kind": "grad", "gen": "rmat", "scale": rng.randint(11, 15), "edge": rng.randint(6, 20), "step": 1,
                    "dtype": dtype, "block_rows": block_rows}
        return {"kind": "grad", "gen": "er", "rows": _log(rng, 2000, 200000), "inner": _log(rng, 2000, 200000),
                "cols": _log(rng, 2000, 200000), "deg_a": rng.randint(2, 20), "deg_b": rng.randint(2, 20), "dtype": dtype,
                "block_rows": block_rows}
    if gen == "rows":
        scale = rng.randint(17, 19)
        return {"kind": "product", "gen": "rmat", "scale": scale, "edge": rng.randint(8, 16),
                "step": rng.choice({17: [3, 5, 7], 18: [7, 11, 15, 21], 19: [21, 27, 37]}[scale]), "dtype": dtype, "block_rows": block_rows}
    case = {"kind": rng.choice(["product", "product", "product", "host"]), "dtype": dtype, "block_rows": block_rows}
    if gen == "er":
        rows, a, b = _log(rng, 500, 1500000), rng.randint(2, 24), rng.randint(2, 40)
        rows = int(min(rows, MOST_PRODUCTS / 2 / (a * b)))
        case.update(gen="er", rows=rows, inner=_log(rng, max(500, rows // 8), 1500000),
                    cols=_log(rng, max(500, rows // 8), 1500000), deg_a=a, deg_b=b)
    elif gen == "mesh":
        lo = rng.randint(2, 40)
        hi = lo + rng.randint(1, 50)
        rows = int(min(_log(rng, 700, 1000000), MOST_PRODUCTS / (hi * hi)))
        case.update(gen="mesh", rows=rows, deg_min=lo, deg_max=hi, band=_log(rng, hi, 10 * hi))
    elif gen == "web":
        case.update(gen="web", rows=_log(rng, 3000, 400000), zipf=round(rng.uniform(1.5, 2.3), 3))
    elif gen == "rmat":
        case.update(gen="rmat", scale=rng.randint(9, 15), edge=rng.randint(4, 20), step=1)
    else:
        case.update(gen="skewed", rows=_log(rng, 1000, 60000), deg=round(rng.uniform(4, 40), 2))
        if rng.random() < 0.4:
            case["kind"] = "noalloc"
    if case["kind"] == "host":
        case["block_rows"] = 4096
    return case


# ---- operands ---------------------------------------------------------------------------------
def _members(case):
    """(rows, mean entries per row) of a batch's members."""
    rng = random.Random("%d %d %d" % (case["members"], case["rows_max"], case["deg_max"]))
    return [(_log(rng, case["rows_min"], case["rows_max"]), rng.uniform(case["deg_min"], case["deg_max"]))
            for _ in range(case["members"])]


@functools.lru_cache(maxsize=1)
def _generated(spec):
    """The case's matrices as generated: a list of (A, B) host CSR pairs; B is A for C = A * A."""
    case = dict(spec)
    dt, gen = np.float64 if case["dtype"] == "f64" else np.float32, case["gen"]
    if case["kind"] == "batch":
        return [(dbd_amd.gen_skewed(n, deg, 1.8, seed=2 * i + 1, dtype=dt),
                 dbd_amd.gen_skewed(n, deg, 1.8, seed=2 * i + 2, dtype=dt)) for i, (n, deg) in enumerate(_members(case))]
    if gen == "er":
        return [(dbd_amd.gen_er(case["rows"], case["inner"], min(case["deg_a"], case["inner"]), seed=1, dtype=dt),
                 dbd_amd.gen_er(case["inner"], case["cols"], min(case["deg_b"], case["cols"]), seed=2, dtype=dt))]
    if gen == "skewed":
        return [(dbd_amd.gen_skewed(case["rows"], case["deg"], 1.8, seed=1, dtype=dt),
                 dbd_amd.gen_skewed(case["rows"], case["deg"], 1.8, seed=2, dtype=dt))]
    if case["kind"] == "grad":
        return [(dbd_amd.gen_rmat(case["scale"], case["edge"], seed=1, add_identity=True, row_normalize=True, dtype=dt),
                 dbd_amd.gen_rmat(case["scale"], case["edge"], seed=2, dtype=dt))]
    if gen == "mesh":
        A = dbd_amd.gen_web(case["rows"], 0.0, case["deg_min"], case["deg_max"], case["band"], 1.0, seed=1, dtype=dt)
    elif gen == "web":
        A = dbd_amd.gen_web(case["rows"], zipf_s=case["zipf"], seed=1, dtype=dt)
    else:
        A = dbd_amd.gen_rmat(case["scale"], case["edge"], seed=1, dtype=dt)
        if case["step"] > 1:
            rows = np.arange(0, A.shape[0], case["step"])
            lens = np.diff(A.ptr)[rows]
            ptr = np.concatenate([[0], np.cumsum(lens)])
            at = np.repeat(A.ptr[rows] - ptr[:-1], lens) + np.arange(ptr[-1])
            return [(dbd_amd.CSR(ptr, A.idx[at], A.val[at], (len(rows), A.shape[1])), A)]
    return [(A, A)]


def _variant(M, row, col, rng):
    """M with its rows and columns shifted around by `row` and `col`, and other values of the same kind."""
    r0 = int(M.ptr[row])
    lens = np.roll(np.diff(M.ptr), -row)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    idx = np.roll(M.idx, -r0)
    low = idx < col  # these come last in their rows
    run = np.concatenate([[0], np.cumsum(low)])
    nlow = run[ptr[1:]] - run[ptr[:-1]]
    to = np.arange(M.nnz) + np.where(low, np.repeat(lens - nlow, lens), -np.repeat(nlow, lens))
    out = np.empty_like(idx)
    out[to] = np.where(low, idx + (M.shape[1] - col), idx - col)
    val = np.roll(M.val, -r0) * rng.uniform(0.5, 1.5, M.nnz).astype(M.val.dtype)
    return dbd_amd.CSR(ptr, out, val, M.shape)


def _operands(case, seed):
    """Host operands (A, B) from the seed: the generated matrices with rows, inner index and columns
    shifted around, so every seed's C has as many entries, and new values. B is A for C = A * A."""
    rng = np.random.default_rng(seed)
    pairs = []
    for A, B in _generated(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "block_rows")))):
        row, inner, col = (int(rng.integers(n)) for n in (A.shape[0], A.shape[1], B.shape[1]))
        if B is A:
            A = B = _variant(A, row, row, rng)
        else:
            A, B = _variant(A, row, inner, rng), _variant(B, inner, col, rng)
        pairs.append((A, B))
    return concat(*zip(*pairs))[:2] if case["kind"] == "batch" else pairs[0]


def prepare(case, seed):
    A, B = _operands(case, seed)
    s = {"kind": case["kind"], "case": case}
    tdt = torch.float64 if case["dtype"] == "f64" else torch.float32
    if case["kind"] == "batch":
        s["runner"] = BatchRunner(A, B, block_rows=case["block_rows"])
        return s
    if case["kind"] == "host":
        s.update(A=A, B=B, ctx=dbd_amd.Context(block_rows=case["block_rows"], dtype=case["dtype"]))
        return s
    dA = dbd_amd.DeviceCSR.from_host(A)
    dB = dA if B is A else dbd_amd.DeviceCSR.from_host(B)
    s.update(A=dA, B=dB, dtype=tdt)
    if case["kind"] == "product":
        s["ctx"] = dbd_amd.Context(block_rows=case["block_rows"], dtype=case["dtype"],
                                   stream=torch.cuda.current_stream())
    elif case["kind"] == "noalloc":
        cap = int(np.diff(B.ptr)[A.idx].sum())  # the products bound the entries of C
        s.update(cap=cap, va=dA.view(), vb=dB.view(), Cptr=torch.empty(A.shape[0] + 1, dtype=torch.int64, device="cuda"),
                 Cidx=torch.empty(cap, dtype=torch.int32, device="cuda"), Cval=torch.empty(cap, dtype=tdt, device="cuda"))
    else:
        s.update(a=dA.val.clone().requires_grad_(True), b=dB.val.clone().requires_grad_(True))
    return s


def run(s):
    kind = s["kind"]
    if kind == "product":
        ctx = s["ctx"]
        ctx.set_operands(s["A"], s["B"])
        ctx.plan()
        Cptr = torch.empty(s["A"].shape[0] + 1, dtype=torch.int64, device="cuda")
        nnz = ctx.symbolic(Cptr)
        Cidx = torch.empty(nnz, dtype=torch.int32, device="cuda")
        Cval = torch.empty(nnz, dtype=s["dtype"], device="cuda")
        ctx.numeric(Cptr, Cidx, Cval)
        return Cptr, Cidx, Cval
    if kind == "noalloc":
        nnz = ctypes.c_int64()
        check(dbd_amd.lib.dbd_spgemm_noalloc(ctypes.byref(s["va"]), ctypes.byref(s["vb"]),
                                             torch.cuda.current_stream().cuda_stream, s["Cptr"].data_ptr(),
                                             s["Cidx"].data_ptr(), s["Cval"].data_ptr(), s["cap"], ctypes.byref(nnz)))
        return s["Cptr"], s["Cidx"][:nnz.value], s["Cval"][:nnz.value]
    if kind == "grad":
        A, B = s["A"], s["B"]
        c, Cptr, Cidx = spgemm_values(A.ptr, A.idx, s["a"], A.shape, B.ptr, B.idx, s["b"], B.shape,
                                      block_rows=s["case"]["block_rows"])
        da, db = torch.autograd.grad(c, (s["a"], s["b"]), grad_outputs=c.detach())
        return Cptr, Cidx, c.detach(), da, db
    if kind == "batch":
        r = s["runner"]
        r.launch()
        return r.Cptr, r.Cidx, r.Cval
    ctx = s["ctx"]
    ctx.set_operands(s["A"], s["B"])
    ctx.run("d2h")
    v = ctx.result_view()  # C where the library put it: pinned host memory, owned by the context

    def array(at, n, ctype):
        view = (ctype * n).from_address(at)
        view.owner = ctx
        return np.ctypeslib.as_array(view)

    return (array(v.ptr, v.nrows + 1, ctypes.c_int64), array(v.idx, v.nnz, ctypes.c_int32),
            array(v.val, v.nnz, ctypes.c_double if s["case"]["dtype"] == "f64" else ctypes.c_float))


def work(case):
    """Operands read once, C written once; with gradients also C's gradient read and the operands' written."""
    A, B = _operands(case, 0)
    with dbd_amd.Context(dtype=case["dtype"]) as ctx:
        ctx.set_operands(A, B)
        products = ctx.plan()["products"]
        nnz = ctx.symbolic(None)
    v = 8 if case["dtype"] == "f64" else 4
    size = lambda m, n: 8 * (m + 1) + (4 + v) * n  # noqa: E731
    total = size(A.shape[0], A.nnz) + (0 if B is A else size(B.shape[0], B.nnz)) + size(A.shape[0], nnz)
    if case["kind"] == "grad":
        return {"bytes": total + v * (nnz + A.nnz + B.nnz), "flops": 6 * products}
    return {"bytes": total, "flops": 2 * products}


# ---- the same in 64 bits, with plain torch --------------------------------------------------------
def exact(case, seed):
    A, B = _operands(case, seed)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    Aptr, Aidx, Aval = dev(A.ptr), dev(A.idx).long(), dev(A.val).double()
    Bptr, Bidx, Bval = dev(B.ptr), dev(B.idx).long(), dev(B.val).double()
    blen = Bptr[1:] - Bptr[:-1]
    per_entry = blen[Aidx]
    before = torch.zeros(A.nnz + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(per_entry, 0, out=before[1:])
    at_row = before[Aptr].cpu().numpy()
    row_of = torch.repeat_interleave(torch.arange(A.shape[0], device="cuda"), Aptr[1:] - Aptr[:-1])
    grad = case["kind"] == "grad"
    da, db = torch.zeros_like(Aval), torch.zeros_like(Bval)
    vals, r0 = [], 0
    while r0 < A.shape[0]:  # rows in runs of some 6e7 products
        r1 = max(r0 + 1, int(np.searchsorted(at_row, at_row[r0] + 6e7, side="right")) - 1)
        e0, e1 = int(A.ptr[r0]), int(A.ptr[r1])
        ent = torch.repeat_interleave(torch.arange(e0, e1, device="cuda"), per_entry[e0:e1])
        pos = Bptr[Aidx[ent]] + torch.arange(ent.numel(), device="cuda") - (before[ent] - before[e0])
        key, order = torch.sort(row_of[ent] * B.shape[1] + Bidx[pos])
        ent, pos = ent[order], pos[order]
        _, slot = torch.unique_consecutive(key, return_inverse=True)
        n = int(slot[-1]) + 1 if slot.numel() else 0
        c = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, slot, Aval[ent] * Bval[pos])
        if grad:
            g = c[slot]
            da.index_add_(0, ent, g * Bval[pos])
            db.index_add_(0, pos, g * Aval[ent])
        vals.append(c)
        r0 = r1
    c = torch.cat(vals)
    return (None, None, c, da, db) if grad else (None, None, c)
