"""Timing cases of the library: what a program that uses it has it do.

Each case is one pass through the public Python entry points (which add only
argument handling to the C ABI): an SpMV, a preconditioned CG solve in each of
its forms (FP64, mixed precision, a block of right-hand sides, many systems,
forward and adjoint of a weighted graph) and the COO -> CSR conversion in front
of them.  Sizes run from a 60 x 52 grid, where launches and latency count, to
the 256^3 Laplacian that the benchmark solves, odd and uneven ones among them.

listed()           the named cases
draw(rng)          one more case of the same ranges
prepare(case, seed) inputs, plans and preconditioners, on the GPU
run(state)         one pass
work(case)         bytes and flops the pass cannot do without
exact(case, seed)  what run returns, from plain torch in FP64
"""
import math

import numpy as np
import torch

from lap_amd import graph as GR
from lap_amd import io as IO
from lap_amd import solver as S
from lap_amd.problems import chung_lu, grid_laplacian, random_geometric_graph

DEV = "cuda"


# ------------------------------------------------------------------- cases

def listed():
    return [
        # one product with a small matrix, as a program's own iteration calls
        # it: launch and call overhead
        {"name": "spmv_60x52", "op": "spmv", "nx": 60, "ny": 52, "nz": 1, "shift": 1e-4},
        # the same call on a power-law graph: hub rows, gathers from all of x
        {"name": "spmv_power_law_300k", "op": "spmv_power_law", "n": 300007},
        # the reference's CPU-runnable configuration: a latency-bound solve
        {"name": "pcg_jacobi_128x128", "op": "pcg", "prec": "line_jacobi", "nx": 128, "ny": 128,
         "nz": 1, "shift": 1e-4, "tol": 1e-8, "weighted": False, "m": 1, "k": 1},
        # the benchmark's headline solve, the largest system
        {"name": "pcg_jacobi_256x256x256", "op": "pcg", "prec": "line_jacobi", "nx": 256,
         "ny": 256, "nz": 256, "shift": 1e-4, "tol": 1e-10, "weighted": False, "m": 1, "k": 1},
        # FP32 inner iteration with FP64 refinement, sides of no round number
        {"name": "mixed_jacobi_190x203x171", "op": "mixed", "prec": "line_jacobi", "nx": 190,
         "ny": 203, "nz": 171, "shift": 1e-4, "tol": 1e-10},
        # incomplete Cholesky: two triangular solves per iteration
        {"name": "pcg_ichol_128x128x128", "op": "pcg", "prec": "ichol", "nx": 128, "ny": 128,
         "nz": 128, "shift": 1e-4, "tol": 1e-10, "weighted": False, "m": 1, "k": 1},
        # symmetric Gauss-Seidel on a grid with uneven conductances
        {"name": "pcg_gs_std_97x110x83_weighted", "op": "pcg", "prec": "GS_std", "nx": 97,
         "ny": 110, "nz": 83, "shift": 1e-4, "tol": 1e-10, "weighted": True, "m": 1, "k": 1},
        # the SpMV-only Gauss-Seidel sweeps
        {"name": "pcg_gs_it2_121x93x140", "op": "pcg", "prec": "GS_it2", "nx": 121, "ny": 93,
         "nz": 140, "shift": 1e-4, "tol": 1e-10, "weighted": False, "m": 1, "k": 3},
        # many right-hand sides of one matrix
        {"name": "block_96x96x96_k32", "op": "block", "nx": 96, "ny": 96, "nz": 96, "rhs": 32,
         "shift": 1e-4, "tol": 1e-10},
        # many uneven systems in one call
        {"name": "batched_160_grids_to_150", "op": "batched", "systems": 160, "lo": 12, "hi": 150,
         "shift": 1e-4, "tol": 1e-10},
        # a training step through the solver: forward and adjoint solves
        {"name": "adjoint_rgg_150k", "op": "adjoint", "n": 150001, "shift": 1e-4, "tol": 1e-10},
        # a matrix file's entries (lower triangle, file order) to device CSR
        {"name": "coo_to_csr_150x160x170", "op": "coo", "nx": 150, "ny": 160, "nz": 170,
         "shift": 1e-4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "spmv_power_law", "pcg", "pcg", "pcg", "mixed", "block", "batched",
                     "adjoint", "coo"])
    if op == "spmv_power_law":
        return {"op": op, "n": _log(rng, 5000, 400000)}
    if op == "adjoint":
        return {"op": op, "n": _log(rng, 3000, 200000), "shift": 1e-4, "tol": 1e-10}
    if op == "batched":
        return {"op": op, "systems": _log(rng, 20, 300), "lo": rng.randint(8, 40),
                "hi": rng.randint(60, 170), "shift": 1e-4, "tol": 1e-10}
    prec = rng.choice(["line_jacobi", "line_jacobi", "ichol", "GS_std", "it_jacobi", "GS_it2"])
    solves = op == "pcg" and prec in ("ichol", "GS_std")  # cost per level of the triangles
    if rng.random() < 0.3 and op not in ("coo", "block"):  # a plane grid
        top = 2500 if op == "spmv" else 160 if solves else 700
        dims = [_log(rng, 40, top), _log(rng, 40, top), 1]
    else:
        top = {"spmv": 220, "pcg": 100 if solves else 150, "mixed": 170, "block": 80,
               "coo": 190}[op]
        dims = [_log(rng, 17, top) for _ in range(3)]
    c = {"op": op, "nx": dims[0], "ny": dims[1], "nz": dims[2], "shift": 1e-4}
    if op in ("spmv", "coo"):
        return c
    c["tol"] = rng.choice([1e-8, 1e-10])
    if op == "block":
        c["rhs"] = rng.choice([4, 8, 16, 32, 64])
        return c
    if op == "mixed":
        c["prec"] = "line_jacobi"
        return c
    c["prec"] = prec
    c["weighted"] = rng.random() < 0.4
    c["m"], c["k"] = 1, {"it_jacobi": 2, "GS_it2": rng.choice([1, 3])}.get(c["prec"], 1)
    return c


# ------------------------------------------------------------------ inputs

def _dims(case):
    return [d for d in (case["nx"], case["ny"], case["nz"]) if d > 1]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _grid_weights(case, seed):
    """Edge weights per axis, laid out like the grid (last axis slowest
    index first); the entry at a point is its edge to the next point."""
    dims = _dims(case)
    shape = dims[::-1]
    g = _gen(seed * 7 + 1)
    out = []
    for ax in range(len(dims)):
        s = list(shape)
        s[len(dims) - 1 - ax] -= 1
        if case.get("weighted"):  # lognormal(0, 1), as the weighted power-law graphs
            out.append(torch.exp(torch.randn(s, dtype=torch.float64, device=DEV, generator=g)))
        else:
            out.append(torch.ones(s, dtype=torch.float64, device=DEV))
    return out


def _grid_csr(case, seed):
    """The grid's graph Laplacian + shift I as CSR arrays on the GPU, rows
    sorted by column (first dimension fastest)."""
    dims = _dims(case)
    nd, shape = len(dims), dims[::-1]
    n = int(np.prod(dims))
    w = _grid_weights(case, seed)
    strides = [1]
    for d in dims[:-1]:
        strides.append(strides[-1] * d)
    full, deg = {}, torch.zeros(shape, dtype=torch.float64, device=DEV)
    for ax in range(nd):
        dim = nd - 1 - ax
        zero = torch.zeros(shape, dtype=torch.float64, device=DEV).narrow(dim, 0, 1)
        full[ax, +1] = torch.cat([w[ax], zero], dim)
        full[ax, -1] = torch.cat([zero, w[ax]], dim)
    idx = torch.arange(n, device=DEV)
    cols, vals, keep = [], [], []
    order = [(ax, -1) for ax in range(nd - 1, -1, -1)] + [None] + [(ax, +1) for ax in range(nd)]
    for o in order:
        if o is not None:
            deg += full[o]
    for o in order:
        if o is None:
            cols.append(idx)
            vals.append(deg.reshape(-1) + case["shift"])
            keep.append(torch.ones(n, dtype=torch.bool, device=DEV))
        else:
            ax, sgn = o
            v = full[o].reshape(-1)
            pos = (idx // strides[ax]) % dims[ax]
            cols.append(idx + sgn * strides[ax])
            vals.append(-v)
            keep.append(pos < dims[ax] - 1 if sgn > 0 else pos > 0)
    keep = torch.stack(keep, 1)
    cols = torch.stack([c.to(torch.int32) for c in cols], 1)
    ja = cols[keep]
    a = torch.stack(vals, 1)[keep]
    ia = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    ia[1:] = torch.cumsum(keep.sum(1), 0).to(torch.int32)
    return n, ia.contiguous(), ja.contiguous(), a.contiguous()


def _matrix(case, seed):
    A = S.DeviceCSR(*_grid_csr(case, seed))
    A.forget()
    return A


def _rhs(n, seed, k=None):
    """b ~ N(0, 1) with its mean taken off, as the benchmark's."""
    shape = (n,) if k is None else (n, k)
    b = torch.randn(shape, dtype=torch.float64, device=DEV, generator=_gen(seed * 7 + 3))
    return b - b.mean(0)


def _coo(case, seed):
    n, ia, ja, a = _grid_csr(case, seed)
    row = torch.repeat_interleave(torch.arange(n, device=DEV), (ia[1:] - ia[:-1]).long())
    low = ja <= row
    rows, cols = row[low].to(torch.int32), ja[low]
    vals = a[low] * (1.0 + 0.1 * torch.rand(int(low.sum()), dtype=torch.float64, device=DEV,
                                            generator=_gen(seed * 7 + 5)))
    return n, rows, cols, vals


def _batch(case, seed):
    """The batch's grids are the program's; the right-hand sides vary by seed."""
    sides = [(int(p), int(q)) for p, q in np.random.default_rng(case["systems"]).integers(
        case["lo"], case["hi"] + 1, (case["systems"], 2))]
    rng = np.random.default_rng(seed)
    return sides, [rng.standard_normal(p * q) for p, q in sides]


def _edge_graph(case, seed):
    """The graph is the program's; weights, b and the target vary by seed."""
    g = random_geometric_graph(case["n"], seed=12345)
    rng = _gen(seed * 7 + 9)
    w = torch.from_numpy(g.w).to(DEV)
    w = w * (0.5 + torch.rand(g.m, dtype=torch.float64, device=DEV, generator=rng))
    b, target = (torch.randn(g.n, dtype=torch.float64, device=DEV, generator=rng)
                 for _ in range(2))
    return g, w, b - b.mean(), target


def prepare(case, seed):
    op = case["op"]
    st = {"op": op, "case": case}
    if op == "spmv_power_law":
        st["A"] = S.DeviceCSR.from_csr(chung_lu(case["n"], seed=seed))
        st["x"] = torch.randn(case["n"], dtype=torch.float64, device=DEV, generator=_gen(seed))
        st["y"] = torch.zeros_like(st["x"])
    elif op == "coo":
        st["n"], st["rows"], st["cols"], st["vals"] = _coo(case, seed)
    elif op == "batched":
        sides, rhs = _batch(case, seed)
        st["B"] = S.Batch.from_systems([grid_laplacian(d, case["shift"]) for d in sides], rhs)
        S.batched_tune(st["B"])  # once per batch, as a program does
    elif op == "adjoint":
        g, st["w"], st["b"], st["target"] = _edge_graph(case, seed)
        st["G"] = GR.GraphLaplacian(g.n, g.src, g.dst, shift=case["shift"])
    else:
        st["A"] = A = _matrix(case, seed)
        st["b"] = _rhs(A.n, seed, case.get("rhs"))
        if op == "spmv":
            st["y"] = torch.zeros_like(st["b"])
        else:  # (the matrix is split on the device: no host copy is read)
            st["P"] = S.make_preconditioner(A, None, case.get("prec", "line_jacobi"),
                                            case.get("m", 1), case.get("k", 1))
    return st


def run(st):
    op, case = st["op"], st["case"]
    if op == "spmv":
        return S.spmv(st["A"], st["b"], st["y"])
    if op == "spmv_power_law":
        return S.spmv(st["A"], st["x"], st["y"])
    if op == "coo":
        A = IO.coo_to_csr(st["n"], st["rows"], st["cols"], st["vals"], True)
        return {"ia": A.ia, "ja": A.ja, "a": A.a}
    if op == "batched":
        x, _, flags, *_ = S.pcg_batched(st["B"], tol=case["tol"])
        return {"x": x, "flags": flags}
    if op == "adjoint":
        w, b = st["w"].detach().requires_grad_(True), st["b"].detach().requires_grad_(True)
        x = GR.laplacian_solve(st["G"], w, b, tol=case["tol"])
        (0.5 * (x - st["target"]).pow(2).sum()).backward()
        return {"x": x, "dw": w.grad, "db": b.grad}
    if op == "block":
        res = S.pcg_block(st["A"], st["b"], st["P"].keep["d_r"], tol=case["tol"])
        return {"x": res.x, "flags": res.flags}
    res = (S.pcg_mixed if op == "mixed" else S.pcg)(st["A"], st["b"], st["P"], tol=case["tol"])
    return {"x": res.x, "flag": res.flag}


# -------------------------------------------------------------------- work

def _iterations(case):
    """About how many iterations the solve takes: they grow with the longest
    side (counts measured on cubes to 1e-10 and on squares to 1e-8)."""
    side = max(_dims(case))
    plane = len(_dims(case)) == 2
    per = {"line_jacobi": 6.9, "it_jacobi": 4.8, "GS_std": 2.5, "GS_it2": 2.65, "ichol": 2.75}
    f = per[case.get("prec", "line_jacobi")] * (0.75 if plane else 1.0)
    if case["tol"] > 1e-9:
        f *= 0.85
    if case.get("weighted"):
        f *= 1.8
    if case["op"] == "mixed":
        f *= 1.3
    return max(1.0, f * side)


def work(case):
    """Per iteration the matrix, its preconditioner and the iteration's
    vectors (x, r, p, 1/diag) read once and x, r, p written once."""
    op = case["op"]
    if op == "spmv_power_law":
        n, nnz = case["n"], 16.5 * case["n"]
        return {"bytes": 12 * nnz + 4 * n + 16 * n, "flops": 2 * nnz}
    if op == "adjoint":
        n, nnz = case["n"], 11 * case["n"]
        it = 12 * math.sqrt(n)  # both solves
        return {"bytes": it * (12 * nnz + 4 * n + 56 * n) + 40 * nnz, "flops": it * (2 * nnz + 12 * n)}
    if op == "batched":
        side = 0.5 * (case["lo"] + case["hi"])
        n = case["systems"] * side * side
        nnz = 5 * n
        it = 6 * side
        return {"bytes": it * (12 * nnz + 4 * n + 56 * n), "flops": it * (2 * nnz + 12 * n)}
    dims = _dims(case)
    n = int(np.prod(dims))
    nnz = n + 2 * sum(n // d * (d - 1) for d in dims)
    if op == "spmv":
        return {"bytes": 12 * nnz + 4 * n + 16 * n, "flops": 2 * nnz}
    if op == "coo":
        return {"bytes": 16 * (nnz + n) // 2 + 12 * nnz + 4 * n, "flops": 0}
    it = _iterations(case)
    if op == "block":
        k = case["rhs"]
        return {"bytes": it * (12 * nnz + 4 * n + (8 + 48 * k) * n), "flops": it * k * (2 * nnz + 12 * n)}
    if op == "mixed":
        return {"bytes": it * (8 * nnz + 4 * n + 28 * n), "flops": it * (2 * nnz + 12 * n)}
    prec, half = case["prec"], 12 * (nnz + n) // 2 + 4 * n
    sweeps = {"line_jacobi": 0, "ichol": 2, "GS_std": 2, "it_jacobi": 2 * (case["k"] - 1),
              "GS_it2": 4 + 2 * case["k"]}[prec]
    return {"bytes": it * (12 * nnz + 4 * n + 56 * n + sweeps * half),
            "flops": it * (2 * nnz + 12 * n + sweeps * (nnz + n))}


# ------------------------------------------------------------------- exact

def _cosine(d):
    """Orthonormal eigenvectors (columns) and eigenvalues of a path graph."""
    i = torch.arange(d, dtype=torch.float64, device=DEV)
    V = torch.cos(math.pi * (i[:, None] + 0.5) * i[None, :] / d) * math.sqrt(2.0 / d)
    V[:, 0] = math.sqrt(1.0 / d)
    return V, 2.0 - 2.0 * torch.cos(math.pi * i / d)


def _grid_solve(dims, shift, b):
    """(L + shift I)^-1 b of an unweighted grid, through its cosine basis; b
    is (n,) or (n, k)."""
    shape = list(dims[::-1])
    x = b.reshape(shape + [-1])
    lam = torch.zeros(shape, dtype=torch.float64, device=DEV) + shift
    bases = []
    for dim, d in enumerate(shape):
        V, ev = _cosine(d)
        bases.append(V)
        lam = lam + ev.reshape([-1 if i == dim else 1 for i in range(len(shape))])
    for back in (False, True):
        for dim, V in enumerate(bases):
            x = torch.movedim(torch.tensordot(V if back else V.T, x, dims=([1], [dim])), 0, dim)
        if not back:
            x = x / lam[..., None]
    return x.reshape(b.shape)


def _edge_solve(n, src, dst, w, shift, b):
    """(L(w) + shift I)^-1 b by Jacobi CG in FP64 run to its rounding level."""
    src, dst = src.long(), dst.long()
    deg = torch.zeros(n, dtype=torch.float64, device=DEV)
    deg.index_add_(0, src, w).index_add_(0, dst, w)

    def mul(x):
        f = w * (x[src] - x[dst])
        y = shift * x
        return y.index_add_(0, src, f).index_add_(0, dst, -f)

    dr = 1.0 / (deg + shift)
    x = torch.zeros_like(b)
    for _ in range(3):  # restarted on the true residual
        r = b - mul(x)
        z = dr * r
        p, rz = z.clone(), torch.dot(r, z)
        stop = 1e-14 * float(b.norm())
        for it in range(20000):
            q = mul(p)
            alpha = rz / torch.dot(p, q)
            x = x + alpha * p
            r = r - alpha * q
            z = dr * r
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
            if it % 50 == 49 and float(r.norm()) < stop:
                break
    return x


def exact(case, seed):
    op = case["op"]
    if op in ("spmv", "spmv_power_law"):
        if op == "spmv":
            n, ia, ja, a = _grid_csr(case, seed)
            x = _rhs(n, seed)
        else:
            M = chung_lu(case["n"], seed=seed)
            n, ia, ja, a = M.n, *(torch.from_numpy(v).to(DEV) for v in (M.ia, M.ja, M.a))
            x = torch.randn(n, dtype=torch.float64, device=DEV, generator=_gen(seed))
        row = torch.repeat_interleave(torch.arange(n, device=DEV), (ia[1:] - ia[:-1]).long())
        return torch.zeros_like(x).index_add_(0, row, a * x[ja.long()])
    if op == "coo":
        n, rows, cols, vals = _coo(case, seed)
        off = rows != cols
        r = torch.cat([rows, cols[off]]).long()
        c = torch.cat([cols, rows[off]]).long()
        order = torch.argsort(r * n + c)
        ia = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
        ia[1:] = torch.cumsum(torch.bincount(r, minlength=n), 0).to(torch.int32)
        return {"ia": ia, "ja": c[order].to(torch.int32),
                "a": torch.cat([vals, vals[off]])[order]}
    if op == "batched":
        sides, rhs = _batch(case, seed)
        x = [_grid_solve(d, case["shift"], torch.from_numpy(b).to(DEV))
             for d, b in zip(sides, rhs)]
        return {"x": torch.cat(x), "flags": None}
    if op == "adjoint":
        g, w, b, target = _edge_graph(case, seed)
        src, dst = (torch.from_numpy(v).to(DEV).long() for v in (g.src, g.dst))
        x = _edge_solve(g.n, src, dst, w, case["shift"], b)
        lam = _edge_solve(g.n, src, dst, w, case["shift"], x - target)
        return {"x": x, "dw": -(lam[src] - lam[dst]) * (x[src] - x[dst]), "db": lam}
    n = int(np.prod(_dims(case)))
    b = _rhs(n, seed, case.get("rhs"))
    if not case.get("weighted"):
        x = _grid_solve(_dims(case), case["shift"], b)
    else:
        idx = torch.arange(n, device=DEV).reshape(_dims(case)[::-1])
        ws = _grid_weights(case, seed)
        src, dst = [], []
        for ax, w in enumerate(ws):
            dim = len(ws) - 1 - ax
            src.append(idx.narrow(dim, 0, idx.shape[dim] - 1).reshape(-1))
            dst.append(idx.narrow(dim, 1, idx.shape[dim] - 1).reshape(-1))
        x = _edge_solve(n, torch.cat(src), torch.cat(dst), torch.cat([w.reshape(-1) for w in ws]),
                        case["shift"], b)
    return {"x": x, "flags" if op == "block" else "flag": None}
