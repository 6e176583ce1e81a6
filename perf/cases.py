"""The work whose speed matters to a user of this library, as cases that can be timed.

Each case is one pass of a program that keeps its matrix (and what it has
prepared of it) on the GPU: products forward and adjoint, gradient passes,
batches, dense tiles, and the first use of a new matrix. The sizes are those
of the benchmark and of the tests, from a 4096-row stencil, where the cost of
a call counts, to the 1.56e9-entry Zipf matrix. Inputs are made with torch
from the seed alone; `exact` computes the same results in 64 bits with plain
torch.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "distributed-ranges_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import drx  # noqa: E402

DEV = "cuda"
DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16,
          "f16": torch.float16}
ITYPES = {"i32": torch.int32, "i64": torch.int64}
CHUNK = 1 << 26  # entries handled at once while inputs are made


def listed():
    return [
        # The smallest calls: a product and an adjoint of a 4096-row stencil,
        # as an iterative solver on a coarse grid issues them.
        {"name": "stencil2d_tiny_f64", "kind": "stencil", "dim": 2, "g": 64, "vdtype": "f64",
         "adjoint": True},
        # An ordinary stencil product (5-point, 1000 x 1000).
        {"name": "stencil2d_f64", "kind": "stencil", "dim": 2, "g": 1000, "vdtype": "f64",
         "adjoint": False},
        # A large stencil with 16-bit storage (7-point, 256^3): values and x
        # in BF16, sums in FP32.
        {"name": "stencil3d_bf16", "kind": "stencil", "dim": 3, "g": 256, "vdtype": "bf16",
         "adjoint": False},
        # A training step through autograd: forward, gradient of the values
        # and gradient of x, over 33 diagonals.
        {"name": "band_train_f32", "kind": "train", "n": 4_000_000, "hw": 16, "vdtype": "f32"},
        # A least-squares gradient: residual and gradient of the values in one
        # fused pass, then the adjoint of the residual from stored CSC values.
        {"name": "band_fused_f32", "kind": "fused", "n": 4_000_000, "hw": 16, "vdtype": "f32"},
        # The largest: irregular rows and columns over an x beyond the caches,
        # through a plan with column panels.
        {"name": "zipf_f32", "kind": "panels", "m": 16_000_000, "n": 16_000_000,
         "vdtype": "f32"},
        # The same kind with 16-bit storage, fewer columns and an odd height.
        {"name": "zipf_bf16", "kind": "panels", "m": 1_000_003, "n": 4_000_000,
         "vdtype": "bf16"},
        # Eight right-hand sides over a wide band, FP64 values and 64-bit
        # indices (what the reference's own gemv benchmark multiplies).
        {"name": "wideband_k8_f64", "kind": "wideband", "n": 50_000, "hw": 1000, "k": 8,
         "vdtype": "f64", "itype": "i64"},
        # Many independent matrices of uneven size, forward and adjoint items
        # in one launch, replayed from a graph: one and sixteen right-hand
        # sides.
        {"name": "batch_k1_f32", "kind": "batch", "nmat": 96, "rows": 200_000, "k": 1},
        {"name": "batch_k16_f32", "kind": "batch", "nmat": 96, "rows": 200_000, "k": 16},
        # A dense tile product c += a b with ragged sizes.
        {"name": "gemm_ragged_f32", "kind": "gemm", "m": 4099, "n": 3001, "k": 2050,
         "vdtype": "f32"},
        # A new matrix: plan, first product, transposed structure and first
        # adjoint (a mesh or a sparsity pattern that has just changed).
        {"name": "new_matrix_f32", "kind": "setup", "m": 600_000, "n": 600_000, "lmin": 3,
         "lmax": 64, "vdtype": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stencil", "stencil", "train", "fused", "panels", "panels", "wideband",
                       "batch", "batch", "gemm", "gemm", "setup"])
    if kind == "stencil":
        dim = rng.choice([2, 3])
        return {"kind": kind, "dim": dim, "g": _log(rng, 32, 1400) if dim == 2 else
                _log(rng, 16, 256), "vdtype": rng.choice(list(DTYPES)),
                "adjoint": rng.random() < 0.4}
    if kind in ("train", "fused"):
        return {"kind": kind, "n": _log(rng, 20_000, 3_000_000), "hw": rng.randint(2, 20),
                "vdtype": rng.choice(["f32", "f32", "f64"])}
    if kind == "panels":
        vdtype = rng.choice(["f32", "f32", "bf16", "f16", "f64"])
        hi = 6_000_000 if vdtype == "f64" else 12_000_000
        return {"kind": kind, "m": _log(rng, 300_000, hi), "n": _log(rng, 2_200_000, hi),
                "vdtype": vdtype}
    if kind == "wideband":
        vdtype = rng.choice(["f64", "f32"])
        return {"kind": kind, "n": _log(rng, 5_000, 50_000), "hw": _log(rng, 100, 1000),
                "k": rng.randint(2, 16), "vdtype": vdtype,
                "itype": rng.choice(["i32", "i64"])}
    if kind == "batch":
        return {"kind": kind, "nmat": _log(rng, 6, 96), "rows": _log(rng, 20_000, 200_000),
                "k": rng.choice([1, 1, 2, 4, 8, 16])}
    if kind == "gemm":
        return {"kind": kind, "m": _log(rng, 96, 5000), "n": _log(rng, 96, 5000),
                "k": _log(rng, 96, 5000), "vdtype": rng.choice(["f32", "f64"])}
    lmin = rng.randint(1, 8)
    return {"kind": kind, "m": _log(rng, 10_000, 600_000), "n": _log(rng, 10_000, 600_000),
            "lmin": lmin, "lmax": lmin + _log(rng, 4, 56), "vdtype": rng.choice(["f32", "f64"])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(n, dtype, g):
    """n values of U[-1, 1)."""
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    shape = n if isinstance(n, tuple) else (n,)
    return (torch.rand(shape, dtype=wide, device=DEV, generator=g) * 2 - 1).to(dtype)


def _normal(n, dtype, g):
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    return torch.randn(n, dtype=wide, device=DEV, generator=g).to(dtype)


def _rowptr(lens, itype):
    rp = torch.zeros(lens.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(lens, 0, out=rp[1:])
    return rp.to(itype)


def _row_chunks(rowptr):
    """Row ranges of about CHUNK entries."""
    rp = rowptr.cpu().to(torch.int64)
    m, r = rp.numel() - 1, 0
    while r < m:
        e = int(torch.searchsorted(rp, int(rp[r]) + CHUNK, right=True)) - 1
        e = min(m, max(e, r + 1))
        yield r, e, int(rp[r]), int(rp[e])
        r = e


def _rows_of(rowptr, r0, r1):
    """Row of every entry of rows [r0, r1), relative to r0, and its row's first entry."""
    rp = rowptr[r0:r1 + 1].to(torch.int64)
    lens = rp[1:] - rp[:-1]
    return torch.repeat_interleave(torch.arange(r1 - r0, device=DEV), lens), rp, lens


def _stratified(rowptr, n, itype, g):
    """Sorted distinct columns: a row of L entries takes one uniform column in
    each of L equal strata of [0, n)."""
    out = torch.empty(int(rowptr[-1]), dtype=itype, device=DEV)
    for r0, r1, a, b in _row_chunks(rowptr):
        if a == b:
            continue
        rows, rp, lens = _rows_of(rowptr, r0, r1)
        j = torch.arange(a, b, device=DEV) - rp[rows]
        L = lens[rows]
        lo = j * n // L
        hi = (j + 1) * n // L
        u = torch.rand(b - a, dtype=torch.float32, device=DEV, generator=g)
        out[a:b] = torch.minimum(lo + (u * (hi - lo)).to(torch.int64), hi - 1).to(itype)
    return out


ZETA = 2.6123753486854883  # sum of l ** -1.5 over l >= 1


def _zipf_lens(m, lmax, g):
    """Row lengths of Zipf(1.5); longer rows are cut to lmax entries."""
    cdf = torch.cumsum(torch.arange(1, lmax, dtype=torch.float64, device=DEV) ** -1.5, 0) / ZETA
    u = torch.rand(m, dtype=torch.float64, device=DEV, generator=g)
    return torch.searchsorted(cdf, u) + 1


def _band(n, hw, vdtype, itype, g):
    i = torch.arange(n, device=DEV)
    lo, hi = torch.clamp(i - hw, min=0), torch.clamp(i + hw, max=n - 1)
    rowptr = _rowptr(hi - lo + 1, itype)
    nnz = int(rowptr[-1])
    colind = torch.empty(nnz, dtype=itype, device=DEV)
    for r0, r1, a, b in _row_chunks(rowptr):
        rows, rp, _ = _rows_of(rowptr, r0, r1)
        colind[a:b] = (lo[r0:r1][rows] + torch.arange(a, b, device=DEV) - rp[rows]).to(itype)
    return rowptr, colind, _normal(nnz, vdtype, g)


def _stencil(dim, g, vdtype, gen):
    """5- or 7-point stencil on a g^dim grid; coefficients of a problem with a
    varying material, not constants."""
    n = g ** dim
    i = torch.arange(n, device=DEV)
    offs, keep = [], []
    for d in reversed(range(dim)):
        s = g ** d
        offs.append(-s)
        keep.append((i // s) % g > 0)
    offs.append(0)
    keep.append(torch.ones(n, dtype=torch.bool, device=DEV))
    for d in range(dim):
        s = g ** d
        offs.append(s)
        keep.append((i // s) % g < g - 1)
    mask = torch.stack(keep, 1)
    rowptr = _rowptr(mask.sum(1), torch.int32)
    cols = i[:, None] + torch.tensor(offs, device=DEV)
    colind = cols[mask].to(torch.int32)
    del cols, mask, keep
    return rowptr, colind, _uniform(colind.numel(), vdtype, gen)


def _sum_dtype(vdtype):
    return torch.float64 if vdtype == torch.float64 else torch.float32


def _inputs(case, seed):
    """The arrays of a case (nothing of the library's): a dict, or a list of
    them for a batch."""
    g, kind = _gen(seed), case["kind"]
    if kind == "batch":
        # the sizes belong to the case, the entries to the seed
        sizes = torch.Generator().manual_seed(case["nmat"] + case["rows"])
        rows = torch.randint(1000, case["rows"] + 1, (case["nmat"],), generator=sizes).tolist()
        out = []
        for m in rows:
            lens = torch.randint(3, 65, (m,), device=DEV, generator=g)
            rowptr = _rowptr(lens, torch.int32)
            k = case["k"]
            shape = (m,) if k == 1 else (k, m)
            out.append({"rowptr": rowptr, "colind": _stratified(rowptr, m, torch.int32, g),
                        "vals": _normal(int(rowptr[-1]), torch.float32, g), "shape": (m, m),
                        "x": _uniform(shape, torch.float32, g),
                        "dy": _uniform(shape, torch.float32, g)})
        return out
    vdtype = DTYPES[case["vdtype"]]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": _uniform((m, k), vdtype, g), "b": _uniform((k, n), vdtype, g),
                "c": _uniform((m, n), vdtype, g)}
    if kind == "stencil":
        rowptr, colind, vals = _stencil(case["dim"], case["g"], vdtype, g)
        m = n = case["g"] ** case["dim"]
    elif kind in ("train", "fused", "wideband"):
        m = n = case["n"]
        rowptr, colind, vals = _band(n, case["hw"], vdtype, ITYPES[case.get("itype", "i32")], g)
    else:
        m, n = case["m"], case["n"]
        lens = _zipf_lens(m, 4096, g) if kind == "panels" else torch.randint(
            case["lmin"], case["lmax"] + 1, (m,), device=DEV, generator=g)
        rowptr = _rowptr(lens, torch.int32)
        colind = _stratified(rowptr, n, torch.int32, g)
        vals = _normal(colind.numel(), vdtype, g)
    d = {"rowptr": rowptr, "colind": colind, "vals": vals, "shape": (m, n)}
    k = case.get("k", 1)
    d["x"] = _uniform(n if k == 1 else (k, n), vdtype, g)
    if kind in ("train", "setup") or case.get("adjoint"):
        d["dy"] = _uniform(m, _sum_dtype(vdtype), g)
    if kind == "fused":
        d["t"] = _uniform(m, vdtype, g)
    return d


# ---------------------------------------------------------------------------
# The passes
# ---------------------------------------------------------------------------
def _matrix(d):
    return drx.CsrMatrix(d["rowptr"], d["colind"], d["vals"], d["shape"])


def prepare(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "batch":
        mats = [_matrix(e) for e in d]
        for A in mats:
            A.set_transposed_values()
        ys = [torch.empty_like(e["x"]) for e in d]
        dxs = [torch.empty_like(e["dy"]) for e in d]
        b = drx.Batch(forward=[(A, e["x"], y) for A, e, y in zip(mats, d, ys)],
                      adjoint=[(A, e["dy"], dx) for A, e, dx in zip(mats, d, dxs)],
                      k=case["k"])
        b.graph()
        # the 64 outputs that may be returned: the largest matrices'
        order = sorted(range(len(d)), key=lambda i: -d[i]["shape"][0])[:32]
        return {"kind": kind, "batch": b, "out": [ys[i] for i in order] +
                [dxs[i] for i in order]}
    state = {"kind": kind, **d}
    if kind in ("gemm", "setup"):
        return state
    state["A"] = A = _matrix(d)
    if kind == "panels":
        A.set_panels()
    if kind == "train":
        state["vals"] = d["vals"].requires_grad_()
        state["x"] = d["x"].requires_grad_()
        A.transpose()
    if kind == "fused":
        A.set_transposed_values()
    if case.get("adjoint"):
        A.transpose()
        # 16-bit values take x in their own type; the adjoint takes dy so too
        state["dy"] = d["dy"].to(d["vals"].dtype)
    return state


def run(state):
    kind = state["kind"]
    if kind == "batch":
        state["batch"].graph_launch()
        return state["out"]
    if kind == "gemm":
        return drx.gemm(state["a"], state["b"], state["c"].clone())
    if kind == "setup":
        A = _matrix(state)
        y = A.matvec(state["x"])
        dx = A.rmatvec(state["dy"])
        A.close()
        return y, dx
    A = state["A"]
    if kind == "train":
        y = drx.spmv(A, state["x"], state["vals"])
        dvals, dx = torch.autograd.grad(y, (state["vals"], state["x"]), state["dy"])
        return y.detach(), dvals, dx
    if kind == "fused":
        y, r, dvals = A.fused_residual(state["x"], state["t"])
        return y, r, dvals, A.rmatvec(r)
    y = A.matvec(state["x"])
    if "dy" in state:
        return y, A.rmatvec(state["dy"])
    return y


# ---------------------------------------------------------------------------
# Work and exact results
# ---------------------------------------------------------------------------
def _size(dtype):
    return torch.empty(0, dtype=dtype).element_size()


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s = _size(DTYPES[case["vdtype"]])
        return {"bytes": s * (m * k + k * n + 3 * m * n), "flops": 2 * m * n * k}
    if kind == "batch":
        m = case["nmat"] * (1000 + case["rows"]) / 2
        nnz, k = m * 33.5, case["k"]
        return {"bytes": 2 * (8 * nnz + 4 * m + 8 * k * m), "flops": 4 * nnz * k}
    vdtype = DTYPES[case["vdtype"]]
    sv, sy = _size(vdtype), _size(_sum_dtype(vdtype))
    si, k = _size(ITYPES[case.get("itype", "i32")]), case.get("k", 1)
    if kind == "stencil":
        dim, g = case["dim"], case["g"]
        m = n = g ** dim
        nnz = (2 * dim + 1) * m - 2 * dim * g ** (dim - 1)
    elif kind in ("train", "fused", "wideband"):
        m = n = case["n"]
        nnz = n * (2 * case["hw"] + 1) - case["hw"] * (case["hw"] + 1)
    else:
        m, n = case["m"], case["n"]
        if kind == "panels":
            p = torch.arange(1, 4096, dtype=torch.float64) ** -1.5 / ZETA
            nnz = m * float((p * torch.arange(1, 4096)).sum() + 4096 * (1 - p.sum()))
        else:
            nnz = m * (case["lmin"] + case["lmax"]) / 2
    product = nnz * (sv + si) + si * (m + 1) + k * (sv * n + sy * m)
    flops = 2 * nnz * k
    if kind == "train":  # forward; dvals; adjoint
        return {"bytes": 2 * product + nnz * (si + sv) + sv * (n + m), "flops": 5 * nnz}
    if kind == "fused":  # forward with t and r, dvals written; adjoint
        return {"bytes": 2 * product + nnz * sv + 2 * sv * m, "flops": 5 * nnz}
    if kind == "setup" or case.get("adjoint"):
        return {"bytes": 2 * product, "flops": 2 * flops}
    return {"bytes": product, "flops": flops}


def _mul(d, x, vals):
    """A x in 64 bits; x is (n,) or (k, n)."""
    x = x.double()
    y = torch.zeros(x.shape[:-1] + (d["shape"][0],), dtype=torch.float64, device=DEV)
    for r0, r1, a, b in _row_chunks(d["rowptr"]):
        rows, _, _ = _rows_of(d["rowptr"], r0, r1)
        c, v = d["colind"][a:b].long(), vals[a:b].double()
        if x.dim() == 1:
            y[r0:r1].index_add_(0, rows, v * x[c])
        else:
            for j in range(x.shape[0]):
                y[j, r0:r1].index_add_(0, rows, v * x[j][c])
    return y


def _mul_t(d, dy, vals):
    dy = dy.double()
    dx = torch.zeros(dy.shape[:-1] + (d["shape"][1],), dtype=torch.float64, device=DEV)
    for r0, r1, a, b in _row_chunks(d["rowptr"]):
        rows, _, _ = _rows_of(d["rowptr"], r0, r1)
        c, v = d["colind"][a:b].long(), vals[a:b].double()
        if dy.dim() == 1:
            dx.index_add_(0, c, v * dy[r0:r1][rows])
        else:
            for j in range(dy.shape[0]):
                dx[j].index_add_(0, c, v * dy[j, r0:r1][rows])
    return dx


def _outer(d, dy, x):
    """dy[row(e)] * x[col(e)] in 64 bits."""
    out = torch.empty(d["colind"].numel(), dtype=torch.float64, device=DEV)
    for r0, r1, a, b in _row_chunks(d["rowptr"]):
        rows, _, _ = _rows_of(d["rowptr"], r0, r1)
        out[a:b] = dy[r0:r1].double()[rows] * x.double()[d["colind"][a:b].long()]
    return out


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "batch":
        order = sorted(range(len(d)), key=lambda i: -d[i]["shape"][0])[:32]
        return ([_mul(d[i], d[i]["x"], d[i]["vals"]) for i in order] +
                [_mul_t(d[i], d[i]["dy"], d[i]["vals"]) for i in order])
    if kind == "gemm":
        return d["c"].double() + d["a"].double() @ d["b"].double()
    y = _mul(d, d["x"], d["vals"])
    if kind == "train":
        return y, _outer(d, d["dy"], d["x"]), _mul_t(d, d["dy"], d["vals"])
    if kind == "fused":
        r = y - d["t"].double()
        return y, r, _outer(d, r, d["x"]), _mul_t(d, r, d["vals"])
    if kind == "setup":
        return y, _mul_t(d, d["dy"], d["vals"])
    if case.get("adjoint"):
        return y, _mul_t(d, d["dy"].to(d["vals"].dtype), d["vals"])
    return y
