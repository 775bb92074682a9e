"""PCG and mixed-precision PCG with the matrix as row classes (the default for large systems with few
distinct rows) against the CSR path: every product and sum is the same, so
solutions, histories and flags are equal bit for bit.  Rows of 1 to 17 entries,
few and too many classes, the first size that is encoded, ragged last row
blocks, an inverse diagonal that does not follow from the row, and infinities.

The CSR path is the one that option spmv_format 1 falls back to when the matrix
has more than 255 distinct values, or the value-indexed one, which is bitwise
the CSR one."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import CSR, grid_laplacian

pytestmark = pytest.mark.gpu

MIN_ROWS = 1 << 19


def band(n, offs, weights=None, shift=0.05):
    """Graph Laplacian + shift of the graph i -- i + o (o in offs), by columns."""
    i = np.arange(n, dtype=np.int64)
    rows, cols, vals = [i], [i], [np.full(n, shift)]
    for k, o in enumerate(offs):
        w = np.ones(n - o) if weights is None else weights(i[: n - o], k)
        lo, hi = i[: n - o], i[o:]
        rows += [lo, hi]
        cols += [hi, lo]
        vals += [-w, -w]
        vals[0][:n - o] += w
        vals[0][o:] += w
    rows, cols, vals = map(np.concatenate, (rows, cols, vals))
    order = np.lexsort((cols, rows))
    ia = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return CSR(n, ia, cols[order].astype(np.int32), vals[order])


def both(Ah, kind, b, maxit=40, d=None, x0=None, solve=None, tol=0.0,
         mk=(1, 1), **opts):
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, kind, *mk)
    if d is not None:
        P.keep["d_r"].copy_(S.to_dev(d))
    out = []
    old = {k: S.set_option(k, v) for k, v in opts.items()}
    try:
        for fmt in (0, 1):
            prev = S.set_option("spmv_format", fmt)
            try:
                kw = {} if x0 is None else {"x0": S.to_dev(x0)}
                out.append((solve or S.pcg)(A, S.to_dev(b), P, tol=tol, maxit=maxit, **kw))
            finally:
                S.set_option("spmv_format", prev)
    finally:
        for k, v in old.items():
            S.set_option(k, v)
    return out


def same(r, s):
    assert (r.iterations, r.flag) == (s.iterations, s.flag)
    assert np.array_equal(r.history, s.history, equal_nan=True)
    assert torch.equal(r.x.view(torch.int64), s.x.view(torch.int64))


CASES = {
    "first_encoded": lambda: band(MIN_ROWS, [1, 777]),
    "last_csr": lambda: band(MIN_ROWS - 1, [1, 777]),
    "cube_odd": lambda: grid_laplacian([83, 79, 89], 0.05),
    "plane": lambda: grid_laplacian([1023, 517], 0.05),
    "diagonal": lambda: CSR(MIN_ROWS + 5, np.arange(MIN_ROWS + 6, dtype=np.int32),
                            np.arange(MIN_ROWS + 5, dtype=np.int32),
                            1.0 + np.arange(MIN_ROWS + 5) % 3),
    "row_9": lambda: band(MIN_ROWS + 257, [1, 2, 900, 901]),
    "row_15": lambda: band(MIN_ROWS + 1, [1, 2, 3, 4, 5, 6, 1000]),
    "row_17": lambda: band(MIN_ROWS + 1, [1, 2, 3, 4, 5, 6, 7, 1000]),  # too wide
    "mixed_classes": lambda: band(MIN_ROWS + 99, [1, 512],  # many classes in every wave
                                  lambda i, k: 1.0 + (i * 2654435761 % 97 % 2)),
    "too_many": lambda: band(MIN_ROWS + 99, [1, 512], lambda i, k: 1.0 + (i * 37 + k) % 509),
}


@pytest.mark.parametrize("name", list(CASES))
def test_bitwise_the_csr_solve(name):
    Ah = CASES[name]()
    b = np.random.default_rng(3).standard_normal(Ah.n)
    same(*both(Ah, "line_jacobi", b))


def test_probe_passes_what_the_encoding_refuses():
    """Few classes among the probed rows, many elsewhere."""
    n = MIN_ROWS + 1024
    at = np.arange(1024, dtype=np.int64) * n // 1024
    far = np.ones(n, bool)
    for o in range(-2, 3):
        far[np.clip(at + o, 0, n - 1)] = False
    Ah = band(n, [1], lambda i, k: np.where(far[i], 1.0 + i % 7919, 1.0))
    b = np.random.default_rng(12).standard_normal(n)
    same(*both(Ah, "line_jacobi", b))


@pytest.mark.parametrize("kind", ["none", "it_jacobi", "GS_it2", "ichol"])
def test_other_preconditioners(kind):
    Ah = grid_laplacian([91, 73, 83], 0.05)
    b = np.random.default_rng(4).standard_normal(Ah.n)
    same(*both(Ah, kind, b, maxit=20))


@pytest.mark.parametrize("rows,walk", [(512, 0), (100, 0), (256, 3)])
def test_row_blocks_and_walks(rows, walk):
    Ah = grid_laplacian([81, 83, 85], 0.05)
    b = np.random.default_rng(5).standard_normal(Ah.n)
    same(*both(Ah, "line_jacobi", b, spmv_rows=rows, spmv_walk=walk))


def test_inverse_diagonal_of_its_own():
    """d_r with few values that do not follow the matrix's rows, and with many."""
    Ah = grid_laplacian([90, 80, 85], 0.05)
    rng = np.random.default_rng(6)
    b = rng.standard_normal(Ah.n)
    for d in (0.1 + 0.05 * (np.arange(Ah.n) % 7), rng.uniform(0.1, 0.2, Ah.n)):
        same(*both(Ah, "line_jacobi", b, d=d))


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_not_finite(bad):
    Ah = grid_laplacian([90, 80, 85], 0.05)
    b = np.random.default_rng(7).standard_normal(Ah.n)
    x0 = np.zeros(Ah.n)
    x0[[0, 4321]] = bad
    r, s = both(Ah, "line_jacobi", b, x0=x0, maxit=40)
    assert (r.iterations, r.flag) == (s.iterations, s.flag)
    assert np.array_equal(r.history, s.history, equal_nan=True)
    assert torch.equal(torch.isnan(r.x), torch.isnan(s.x))


@pytest.mark.parametrize("name", ["first_encoded", "cube_odd", "plane", "diagonal", "row_9",
                                  "row_15", "row_17", "mixed_classes", "too_many"])
@pytest.mark.parametrize("vectors", [0, 1])
def test_mixed_bitwise(name, vectors):
    """Also through refinements; rows of 15 entries fill cls_inner's 16."""
    Ah = CASES[name]()
    b = np.random.default_rng(8).standard_normal(Ah.n)
    r, s = both(Ah, "line_jacobi", b, maxit=60, solve=S.pcg_mixed, tol=1e-9,
                mixed_vectors=vectors)
    assert r.refinements == s.refinements and r.refinements > 0
    same(r, s)


@pytest.mark.parametrize("kind", ["none", "ichol"])
def test_mixed_other_preconditioners(kind):
    Ah = grid_laplacian([91, 73, 83], 1e-6)
    b = np.random.default_rng(9).standard_normal(Ah.n)
    same(*both(Ah, kind, b, maxit=25, solve=S.pcg_mixed, tol=1e-8))


def test_mixed_rows_without_a_diagonal():
    """Not positive definite, so few steps: rows of off-diagonals only, up to 16."""
    Ah = band(MIN_ROWS + 3, [1, 2, 3, 4, 5, 6, 7, 900])
    keep = np.ones(Ah.nnz, bool)
    rows = np.repeat(np.arange(Ah.n), np.diff(Ah.ia))
    keep[(rows == Ah.ja) & (rows % 2 == 0)] = False
    keep[(rows == Ah.ja + 900) | (rows + 900 == Ah.ja)] = False
    Bh = CSR(Ah.n, np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=Ah.n))])
             .astype(np.int32), Ah.ja[keep], Ah.a[keep])
    b = np.random.default_rng(10).standard_normal(Bh.n)
    same(*both(Bh, "none", b, maxit=20, solve=S.pcg_mixed, tol=1e-9))


@pytest.mark.parametrize("kind,m,k", [("it_jacobi", 1, 1), ("it_jacobi", 1, 4), ("GS_it", 1, 1),
                                      ("GS_it", 3, 2), ("GS_it2", 1, 1), ("GS_it2", 2, 3)])
@pytest.mark.parametrize("name", ["first_encoded", "cube_odd", "row_9", "row_15", "row_17",
                                  "mixed_classes", "one_sided", "too_many"])
def test_sweeps(kind, m, k, name):
    """Triangles of 2, 3, 4, 7 and 8 entries a row, and of 1 and 14 (so one
    table is as wide as the other needs)."""
    if name == "one_sided":
        Ah = band(MIN_ROWS + 1, [1])
        rows = np.repeat(np.arange(Ah.n), np.diff(Ah.ia))
        ja = np.concatenate([Ah.ja] + [np.arange(Ah.n) - o for o in range(2, 15)])
        rows = np.concatenate([rows, np.tile(np.arange(Ah.n), 13)])
        a = np.concatenate([Ah.a, np.full(13 * Ah.n, -1e-3)])
        keep = ja >= 0
        rows, ja, a = rows[keep], ja[keep], a[keep]
        order = np.lexsort((ja, rows))
        Ah = CSR(Ah.n, np.concatenate([[0], np.cumsum(np.bincount(rows))]).astype(np.int32),
                 ja[order].astype(np.int32), a[order])
    else:
        Ah = CASES[name]()
    b = np.random.default_rng(11).standard_normal(Ah.n)
    same(*both(Ah, kind, b, maxit=20, mk=(m, k)))
