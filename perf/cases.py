"""The work that programs have this library do, for timing it: sparse products y = A x with a
resident matrix through each family of schedules, products with several right-hand sides, the
conjugate gradient solver, the learned choice of a schedule with everything that a new matrix
costs, and the host-pointer call sequence of a program written against the reference's API.

A case is a dict of plain values. `prepare` makes its inputs on the GPU from the seed and the
handles that a program keeps between calls; `run` is one pass through the public entry points.

  op       spmv    y = A x: the column order applied to a new x, then one product
           spmm    Y = A X, X with k columns, row by row
           build   a new matrix: features, schedule choice, layout, schedule, first product
           cg      one solve
           host    csr_to_csc, ColSort, formatTransform and FastLoad_spmv on host arrays
  pattern  bus       structurally symmetric, full diagonal, short columns (power networks)
           grid27    27-point stencil on an n^3 grid
           zipf      column lengths Zipf(`shape`) up to 50,000, rows anywhere (graphs, text)
           uniform   about `shape` entries per column, rows anywhere
           blocks    dense-ish diagonal blocks of 512, `shape` entries per column
           batch     n square Zipf(2) matrices of 1,000 to 200,000 rows stacked on the diagonal
"""
import math

import numpy as np
import torch

import fastload_amd as fl
from fastload_amd import selector

KERNELS = {"dropin": fl.KERNEL_DROPIN, "winr": fl.KERNEL_WINR, "pb": fl.KERNEL_PB, "hyb": fl.KERNEL_HYB}
BLOCK = 512       # rows of a diagonal block ("blocks")
ZIPF_MAX = 50000  # longest column ("zipf")


def listed():
    return [
        # the reference's own input size: one small resident product, latency and launches
        {"name": "spmv_bus_f64", "op": "spmv", "pattern": "bus", "n": 1138, "shape": 2.6, "kernel": "dropin", "kind": "f64", "k": 1},
        # a reference-style program end to end on host arrays
        {"name": "host_bus_f64", "op": "host", "pattern": "bus", "n": 60013, "shape": 8.0, "kernel": "dropin", "kind": "f64", "k": 1},
        # a large structured grid, FP32 (the benchmark's second workload)
        {"name": "spmv_grid_f32", "op": "spmv", "pattern": "grid27", "n": 128, "shape": 27.0, "kernel": "winr", "kind": "f32", "k": 1},
        # the benchmark's power-law matrix with its value + slot words
        {"name": "spmv_zipf_packed", "op": "spmv", "pattern": "zipf", "n": 4194304, "shape": 1.8423, "kernel": "hyb", "kind": "packed", "k": 1},
        # a power-law matrix in the reference's precision
        {"name": "spmv_zipf_f64", "op": "spmv", "pattern": "zipf", "n": 1000003, "shape": 1.8423, "kernel": "hyb", "kind": "f64", "k": 1},
        # rows without locality and no long columns
        {"name": "spmv_uniform_f32", "op": "spmv", "pattern": "uniform", "n": 1500007, "shape": 12.0, "kernel": "pb", "kind": "f32", "k": 1},
        # short independent rows, x in the original order (the schedule chosen most often)
        {"name": "spmv_blocks_f32", "op": "spmm", "pattern": "blocks", "n": 524288, "shape": 24.0, "kernel": "row", "kind": "f32", "k": 1},
        # many small matrices at once with a few and with many right-hand sides
        {"name": "spmm_batch_k8_f32", "op": "spmm", "pattern": "batch", "n": 128, "shape": 2.0, "kernel": "row", "kind": "f32", "k": 8},
        {"name": "spmm_batch_k32_f32", "op": "spmm", "pattern": "batch", "n": 64, "shape": 2.0, "kernel": "row", "kind": "f32", "k": 32},
        # a block of vectors on a grid in FP64 (block solvers)
        {"name": "spmm_grid_k16_f64", "op": "spmm", "pattern": "grid27", "n": 64, "shape": 27.0, "kernel": "row", "kind": "f64", "k": 16},
        # a matrix that is new: chosen, prepared and multiplied once
        {"name": "build_zipf_f32", "op": "build", "pattern": "zipf", "n": 600011, "shape": 1.8423, "kernel": "chosen", "kind": "f32", "k": 1},
        # the solver that repeats the product
        {"name": "cg_grid_f64", "op": "cg", "pattern": "grid27", "n": 80, "shape": 27.0, "kernel": "winr", "kind": "f64", "k": 1},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["small", "host", "grid", "zipf", "uniform", "row", "spmm", "spmm", "build", "cg"])
    if op == "small":
        return {"op": "spmv", "pattern": "bus", "n": _size(rng, 300, 30000), "shape": round(rng.uniform(1.5, 8.0), 2),
                "kernel": "dropin", "kind": rng.choice(["f64", "f64", "f32"]), "k": 1}
    if op == "host":
        return {"op": "host", "pattern": "bus", "n": _size(rng, 500, 60000), "shape": round(rng.uniform(1.5, 8.0), 2),
                "kernel": "dropin", "kind": "f64", "k": 1}
    if op == "grid":
        return {"op": "spmv", "pattern": "grid27", "n": _size(rng, 22, 127), "shape": 27.0, "kernel": "winr",
                "kind": rng.choice(["f32", "f64", "packed", "bf16x2"]), "k": 1}
    if op == "zipf":
        return {"op": "spmv", "pattern": "zipf", "n": _size(rng, 60000, 3000000), "shape": round(rng.uniform(1.75, 2.3), 4),
                "kernel": "hyb", "kind": rng.choice(["f32", "f64", "packed"]), "k": 1}
    if op == "uniform":
        return {"op": "spmv", "pattern": "uniform", "n": _size(rng, 100000, 3000000), "shape": round(rng.uniform(3.0, 12.0), 2),
                "kernel": "pb", "kind": rng.choice(["f32", "f64", "packed"]), "k": 1}
    if op == "row":
        return {"op": "spmm", "pattern": rng.choice(["blocks", "uniform"]), "n": _size(rng, 40000, 800000),
                "shape": round(rng.uniform(3.0, 32.0), 2), "kernel": "row", "kind": rng.choice(["f32", "f64"]), "k": 1}
    if op == "spmm":
        pattern = rng.choice(["batch", "batch", "grid27", "blocks", "zipf"])
        n, shape = {"batch": (_size(rng, 8, 60), 2.0), "grid27": (_size(rng, 30, 72), 27.0),
                    "blocks": (_size(rng, 40000, 300000), round(rng.uniform(4.0, 32.0), 2)),
                    "zipf": (_size(rng, 60000, 400000), round(rng.uniform(1.8, 2.3), 4))}[pattern]
        return {"op": "spmm", "pattern": pattern, "n": n, "shape": shape, "kernel": "row",
                "kind": rng.choice(["f32", "f32", "f64"]), "k": rng.choice([2, 4, 8, 8, 16, 32])}
    if op == "build":
        pattern = rng.choice(["zipf", "uniform", "blocks", "grid27"])
        n, shape = {"zipf": (_size(rng, 50000, 600000), round(rng.uniform(1.8, 2.3), 4)),
                    "uniform": (_size(rng, 50000, 800000), round(rng.uniform(3.0, 12.0), 2)),
                    "blocks": (_size(rng, 20000, 300000), round(rng.uniform(4.0, 32.0), 2)),
                    "grid27": (_size(rng, 22, 70), 27.0)}[pattern]
        return {"op": "build", "pattern": pattern, "n": n, "shape": shape, "kernel": "chosen", "kind": "f32", "k": 1}
    return {"op": "cg", "pattern": "grid27", "n": _size(rng, 22, 79), "shape": 27.0,
            "kernel": rng.choice(["winr", "row"]), "kind": "f64", "k": 1}


# ------------------------------------------------------------------------------- matrices
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _zipf_lengths(count, exponent, longest, g):
    """Lengths at the quantiles of Zipf(exponent) on 1..longest, in random order."""
    p = torch.arange(1, longest + 1, device="cuda", dtype=torch.float64) ** -exponent
    cdf = torch.cumsum(p, 0)
    q = (torch.arange(count, device="cuda", dtype=torch.float64) + 0.5) / count * cdf[-1]
    return (torch.searchsorted(cdf, q) + 1).clamp_(max=longest)[torch.randperm(count, device="cuda", generator=g)]


def _batch_sizes(count):
    rng = np.random.default_rng(512)
    return np.exp(rng.uniform(math.log(1e3), math.log(2e5), int(count))).astype(np.int64)


def _spread(lengths, first, height, g):
    """CSC whose column c has lengths[c] distinct ascending rows in [first, first + height): one
    uniform row in each of lengths[c] equal parts of the range."""
    colptr = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=colptr[1:])
    nnz = int(colptr[-1])
    col = torch.repeat_interleave(torch.arange(lengths.numel(), device="cuda"), lengths, output_size=nnz)
    j = torch.arange(nnz, device="cuda") - colptr[col]
    size = lengths[col]
    tall = height[col] if isinstance(height, torch.Tensor) else height
    lo = j * tall // size
    part = (j + 1) * tall // size - lo
    u = torch.rand(nnz, device="cuda", generator=g, dtype=torch.float64)
    row = lo + torch.minimum((u * part).to(torch.int64), part - 1)
    if isinstance(first, torch.Tensor):
        row += first[col]
    return colptr.to(torch.int32), row.to(torch.int32)


def _matrix(case, seed):
    """(m, n, colptr, rowidx, val): int32, int32 and float64 tensors on the GPU."""
    g, pattern, n, shape = _gen(seed), case["pattern"], int(case["n"]), float(case["shape"])
    if pattern == "grid27":
        side, n = n, n ** 3
        c = torch.arange(n, device="cuda", dtype=torch.int32)
        x, y, z = c % side, c // side % side, c // (side * side)
        keep, row = [], []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    keep.append((x + dx >= 0) & (x + dx < side) & (y + dy >= 0) & (y + dy < side) & (z + dz >= 0) & (z + dz < side))
                    row.append(c + (dz * side + dy) * side + dx)
        keep, row = torch.stack(keep, 1), torch.stack(row, 1)
        colptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        torch.cumsum(keep.sum(1), 0, out=colptr[1:])
        if case["op"] == "cg":
            val = torch.where(row == c[:, None], 26.0, -1.0)[keep].double()
            return n, n, colptr.to(torch.int32), row[keep], val
        rowidx = row[keep]
        val = torch.rand(rowidx.numel(), device="cuda", generator=g) + 0.5
        val *= torch.randint(0, 2, val.shape, device="cuda", generator=g) * 2 - 1
        return n, n, colptr.to(torch.int32), rowidx, val.double()
    if pattern == "bus":
        # one network per size, its nodes renumbered by the seed: the layout's sizes do not vary
        fixed = _gen(n)
        a, b = torch.randint(0, n, (2, int(n * shape / 2)), device="cuda", generator=fixed)
        name = torch.randperm(n, device="cuda", generator=g)
        a, b, d = name[a[a != b]], name[b[a != b]], torch.arange(n, device="cuda")
        key = torch.unique(torch.cat([a * n + b, b * n + a, d * n + d]))
        col, row = key // n, key % n
        colptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        torch.cumsum(torch.bincount(col, minlength=n), 0, out=colptr[1:])
        val = torch.rand(key.numel(), device="cuda", generator=g, dtype=torch.float64) * 2 - 1 + 4.0 * (col == row)
        return n, n, colptr.to(torch.int32), row.to(torch.int32), val
    if pattern == "batch":
        sizes = torch.from_numpy(_batch_sizes(n)).cuda()
        n = int(sizes.sum())
        block = torch.repeat_interleave(torch.arange(sizes.numel(), device="cuda"), sizes, output_size=n)
        first, height = (torch.cumsum(sizes, 0) - sizes)[block], sizes[block]
        lengths = torch.minimum(_zipf_lengths(n, shape, 200000, g), height)
        colptr, rowidx = _spread(lengths, first, height, g)
    elif pattern == "blocks":
        n = max(1, n // BLOCK) * BLOCK
        lengths = torch.poisson(torch.full((n,), shape, device="cuda"), generator=g).to(torch.int64).clamp_(1, BLOCK)
        first = torch.arange(n, device="cuda") // BLOCK * BLOCK
        colptr, rowidx = _spread(lengths, first, BLOCK, g)
    elif pattern == "uniform":
        lengths = torch.poisson(torch.full((n,), shape, device="cuda"), generator=g).to(torch.int64)
        colptr, rowidx = _spread(lengths, 0, n, g)
    else:
        lengths = _zipf_lengths(n, shape, min(n, ZIPF_MAX), g)
        colptr, rowidx = _spread(lengths, 0, n, g)
    val = torch.randn(rowidx.numel(), device="cuda", generator=g)  # FP32 data, given to the library in FP64
    return n, n, colptr, rowidx, val.double()


def _vector(case, n, seed):
    double = case["kind"] == "f64"
    return torch.randn(n * int(case["k"]), device="cuda", generator=_gen(seed + 1000003), dtype=torch.float64 if double else torch.float32)


def _expected(case):
    """Rows and about how many entries the case's matrix has."""
    n, shape = int(case["n"]), float(case["shape"])
    if case["pattern"] == "grid27":
        return n ** 3, (3 * n - 2) ** 3
    if case["pattern"] == "bus":
        return n, n * (1 + shape)
    if case["pattern"] == "batch":
        sizes = _batch_sizes(n)
        return int(sizes.sum()), sum(s * (math.log(s) + 1.6) for s in sizes) * 6 / math.pi ** 2
    if case["pattern"] in ("uniform", "blocks"):
        return n, n * shape
    k = np.arange(1, min(n, ZIPF_MAX) + 1, dtype=np.float64)
    return n, n * float((k ** (1 - shape)).sum() / (k ** -shape).sum())


# ------------------------------------------------------------------------------ the calls
def _wrap(t):
    """A tensor's memory as the library's device buffer (which does not own it)."""
    d = object.__new__(fl.DeviceArray)
    d.dtype = np.dtype(str(t.dtype).replace("torch.", ""))
    d.count, d.nbytes, d.ptr, d._parent = t.numel(), t.numel() * t.element_size(), t.data_ptr(), t
    return d


def _kind(case):
    return {"f64": fl.VAL_F64, "f32": fl.VAL_F32, "packed": fl.VAL_PACKED, "bf16x2": fl.VAL_BF16X2}[case["kind"]]


def prepare(case, seed):
    m, n, colptr, rowidx, val = _matrix(case, seed)
    op, kind = case["op"], _kind(case)
    if op == "host":  # CSR of the structurally symmetric matrix on the host
        return {"case": case, "m": m, "n": n, "rowptr": colptr.cpu().numpy(), "colidx": rowidx.cpu().numpy(),
                "val": val.cpu().numpy(), "x": _vector(case, n, seed).cpu().numpy()}
    x = _vector(case, n, seed)
    y = torch.empty(m * int(case["k"]), device="cuda", dtype=torch.float64 if kind in (fl.VAL_F64, fl.VAL_BF16X2) else torch.float32)
    s = {"case": case, "m": m, "n": n, "x": x, "y": y, "dx": _wrap(x), "dy": _wrap(y), "kind": kind, "k": int(case["k"])}
    csc = (_wrap(colptr), _wrap(rowidx), _wrap(val))
    if op == "build":
        s.update(csc=csc, chooser=selector.Selector())
        return s
    A = s["A"] = fl.FastLoadMatrix(m, n, *csc, width=32 if case["kernel"] == "dropin" else 64)
    if case["kernel"] == "row":
        A.prepare_rows()
    else:
        s["kernel"] = KERNELS[case["kernel"]]
        if kind != fl.VAL_F64:
            A.prepare(fl.VAL_F32 if kind == fl.VAL_PACKED else kind)
        if case["kernel"] == "winr":
            A.prepare_schedule(fl.KERNEL_WINR, 64, 0)
        elif case["kernel"] == "pb":
            A.prepare_schedule(fl.KERNEL_PB, 128 if kind == fl.VAL_PACKED else 256, 16384)  # packed: room for the slot bits
        elif case["kernel"] == "hyb":
            A.prepare_hyb(min(n, 19456 if kind == fl.VAL_F64 else 32768), 128, 16384)
        if kind == fl.VAL_PACKED:
            A.prepare(kind)
        sx = torch.empty_like(x)
        s.update(sx=sx, dsx=_wrap(sx))
    if op == "cg":
        s["cg"] = fl.CG(A, fl.KERNEL_ROW if case["kernel"] == "row" else s["kernel"], kind)
    return s


def run(s):
    op = s["case"]["op"]
    if op == "spmv":
        s["A"].permute_x(s["dx"], s["dsx"])
        s["A"].spmv(s["dsx"], s["dy"], s["kernel"], s["kind"], assign=True)
        return s["y"]
    if op == "spmm":
        s["A"].spmm(s["dx"], s["dy"], s["k"], s["kind"])
        return s["y"]
    if op == "cg":  # from x = 0
        s["y"].zero_()
        iterations, residual = s["cg"].solve(s["dx"], s["dy"], max_iter=1000, rtol=1e-8, check_every=10)
        return {"x": s["y"], "iterations": iterations, "residual": residual}
    if op == "build":
        cls, probability, features = s["chooser"].choose(s["m"], s["n"], s["csc"][0], s["csc"][1])
        product = selector.ScheduledSpMV(s["m"], s["n"], *s["csc"], cls)
        product.set_x(s["dx"])
        product.step(s["dy"])
        return {"class": cls, "probability": probability, "features": features, "y": s["y"]}
    m, n = s["m"], s["n"]
    val, row, colptr, lengths, _ = fl.csr_to_csc(m, n, s["val"], s["rowptr"], s["colidx"])
    srow, sval, slen, sx, _ = fl.ColSort(m, n, lengths, colptr, row, val, s["x"])
    tiles, levels, _, _ = fl.formatTransform(srow, sval, slen, len(val), m, n)
    y, _, _ = fl.FastLoad_spmv(tiles, len(val), n, m, sx)
    return {"colptr": colptr, "levels": levels, "tile_ptr": tiles.tile_ptr, "rows": tiles.sortrowidx,
            "values": tiles.sortval, "segments": tiles.sortrowindex, "y": y}


# ---------------------------------------------------------------- what the work amounts to
def work(case):
    m, nnz = _expected(case)
    k, op = int(case["k"]), case["op"]
    value = vector = 8 if case["kind"] == "f64" else 4
    out = 8 if case["kind"] in ("f64", "bf16x2") else 4
    product = nnz * (value + 4) + m * k * (vector + out)
    flops = 2.0 * nnz * k
    if op == "cg":  # a product and the vectors x, r, p, q read and x, r, p written, per iteration
        iterations = 2 * int(case["n"])
        return {"bytes": float(iterations * (product + 7 * 8 * m)), "flops": iterations * (flops + 10.0 * m)}
    if op == "build":  # the matrix as it comes (FP64 values), x and y
        return {"bytes": float(nnz * 12 + 4 * m + 8 * m), "flops": flops}
    if op == "host":  # in: CSR and x; out: the layout and y
        return {"bytes": float(nnz * 24 + 20 * m), "flops": 101 * flops}
    return {"bytes": float(product), "flops": flops}


# ------------------------------------------------------------------------ results in FP64
def _product(m, colptr, rowidx, val, x, k):
    """A X for a CSC matrix, in FP64."""
    lengths = (colptr[1:] - colptr[:-1]).to(torch.int64)
    nnz = rowidx.numel()
    col = torch.repeat_interleave(torch.arange(lengths.numel(), device="cuda"), lengths, output_size=nnz)
    X = x.double().view(-1, k)
    Y = torch.zeros(m, k, device="cuda", dtype=torch.float64)
    step = max(1, (1 << 26) // k)
    for i in range(0, nnz, step):
        e = slice(i, i + step)
        Y.index_add_(0, rowidx[e].to(torch.int64), val[e, None] * X[col[e]])
    return Y.view(-1)


def exact(case, seed):
    m, n, colptr, rowidx, val = _matrix(case, seed)
    x, op, k = _vector(case, n, seed), case["op"], int(case["k"])
    if op == "cg":
        return _exact_cg(case, x)
    y = _product(m, colptr, rowidx, val, x, k)
    if op == "build":
        return {"class": None, "probability": None, "features": _exact_features(m, n, colptr, rowidx), "y": y}
    if op == "host":  # the prepared arrays are the CSR of A, so the result is that of its transpose
        lengths = (colptr[1:] - colptr[:-1]).to(torch.int64)
        owner = torch.repeat_interleave(torch.arange(n, device="cuda"), lengths)
        y = torch.zeros(m, device="cuda", dtype=torch.float64).index_add_(0, owner, val * x[rowidx.to(torch.int64)])
        return {"colptr": None, "levels": None, "tile_ptr": None, "rows": None, "values": None, "segments": None, "y": y}
    return y


def _exact_cg(case, b):
    """The solver's iterations in FP64: A = 27 I - S, S the sum over the 3 x 3 x 3 neighbourhood."""
    side = int(case["n"])

    def product(v):
        s = v.view(side, side, side)
        for d in range(3):
            t = s.clone()
            t.narrow(d, 1, side - 1).add_(s.narrow(d, 0, side - 1))
            t.narrow(d, 0, side - 1).add_(s.narrow(d, 1, side - 1))
            s = t
        return 27.0 * v - s.reshape(-1)

    x, r = torch.zeros_like(b), b.clone()
    p, rr, norm = r.clone(), float(r @ r), math.sqrt(float(b @ b))
    iterations = 0
    while iterations < 1000:
        least = math.inf
        for _ in range(10):
            q = product(p)
            a = rr / float(p @ q)
            x += a * p
            r -= a * q
            new = float(r @ r)
            p, rr = r + new / rr * p, new
            least = min(least, math.sqrt(rr))
        iterations += 10
        if least / norm <= 1e-8:
            break
    return {"x": x, "iterations": None, "residual": math.sqrt(rr) / norm}


def _exact_features(m, n, colptr, rowidx):
    cp = colptr.to(torch.int64)
    lengths = cp[1:] - cp[:-1]
    nnz = rowidx.numel()
    bins = torch.where(lengths > 0, torch.log2(lengths.double().clamp(min=1)).floor() + 1, 0.0).clamp(max=31).to(torch.int64)
    f = torch.zeros(40, dtype=torch.float64, device="cuda")
    f[:32] = torch.bincount(bins, minlength=32)[:32].double() / n
    rows = torch.bincount(rowidx.to(torch.int64), minlength=m).double()
    mean = rows.mean()
    some = lengths > 0
    span = (rowidx[cp[1:][some] - 1] - rowidx[cp[:-1][some]]).double() / m
    f[32], f[33], f[34] = math.log2(m + 1) / 24, math.log2(n + 1) / 24, math.log2(nnz + 1) / 32
    f[35] = torch.log2(mean + 1) / 8
    f[36] = ((rows * rows).mean() - mean * mean).clamp(min=0).sqrt() / mean
    f[37] = torch.log2(rows.max() / mean + 1) / 8
    f[38] = (rows == 0).double().mean()
    f[39] = span.mean()
    return f
