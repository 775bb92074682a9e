"""Jacobi PCG as one launch (small and medium systems): every row-length class
and its first size past it, one and several workgroups, ragged last workgroups,
rows referred to from far away, a start vector, and every way a solve ends.

The solves run a fixed number of iterations, so the result is compared with the
oracle's after exactly as many: the two sum dot products in different orders,
which the recurrence carries on (relative 1e-16 per iteration, amplified by the
residual's reduction, here at most 1e3); 1e-10 leaves three digits."""
import numpy as np
import pytest
import torch

import oracle
from lap_amd import solver as S
from lap_amd.problems import CSR, from_coo, grid_laplacian

pytestmark = pytest.mark.gpu


def circulant(n, offsets):
    """Weighted circulant graph Laplacian + I/4: rows of 2 len(offsets) + 1
    entries, neighbours up to max(offsets) rows away in both directions."""
    i = np.arange(n)
    rows = np.concatenate([np.maximum(i, (i + o) % n) for o in offsets])
    cols = np.concatenate([np.minimum(i, (i + o) % n) for o in offsets])
    w = 0.5 + (rows * 5 + cols * 3) % 13 / 9.0
    diag = np.bincount(rows, w, n) + np.bincount(cols, w, n) + 0.25
    return from_coo(n, np.concatenate([rows, i]), np.concatenate([cols, i]),
                    np.concatenate([-w, diag]), symmetric=True)


def offsets(m):
    return [1, 2, 600, 1777, 30, 31, 1100][:m] + list(range(40, 40 + max(0, m - 7)))


CASES = {
    "one_row": lambda: grid_laplacian([1], 0.5),
    "two_rows": lambda: grid_laplacian([2], 0.5),
    "line_2049": lambda: grid_laplacian([2049], 0.05),
    "plane_64x32": lambda: grid_laplacian([64, 32], 0.05),  # exactly one workgroup
    "plane_130x90": lambda: grid_laplacian([130, 90], 0.05),
    "cube_23": lambda: grid_laplacian([23, 23, 23], 0.05),
    "diagonal": lambda: CSR(3000, np.arange(3001, dtype=np.int32), np.arange(3000, dtype=np.int32),
                            1.0 + np.arange(3000) % 5),
    **{f"circulant_{2 * m + 1}": (lambda m=m: circulant(5003, offsets(m)))
       for m in (2, 3, 4, 7, 8, 11, 12, 15, 16)},  # 33 entries: three launches an iteration
}


@pytest.mark.parametrize("name", list(CASES))
def test_fixed_iterations_match_the_oracle(name):
    Ah = CASES[name]()
    rng = np.random.default_rng(7)
    b = rng.standard_normal(Ah.n)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    its = 1 if name in ("one_row", "diagonal") else 2 if name == "two_rows" else 12
    res = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=its - 1)
    xo, ito, flo, hist = oracle.Oracle().cg(Ah, b, "line_jacobi", tol=0.0, maxit=its - 1)
    assert (res.iterations, res.flag) == (ito, flo)
    x = res.x.cpu().numpy()
    print(f"[diag] {name}: {np.linalg.norm(x - xo) / np.linalg.norm(xo):.2e}", flush=True)
    assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)
    again = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=its - 1)  # meets the first solve's tags
    assert torch.equal(again.x, res.x) and np.array_equal(again.history, res.history)


def test_start_vector_and_every_end():
    Ah = grid_laplacian([70, 60], 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    rng = np.random.default_rng(8)
    b, x0 = rng.standard_normal(Ah.n), rng.standard_normal(Ah.n)
    full = S.pcg(A, S.to_dev(b), P, tol=1e-12, x0=S.to_dev(x0))
    cold = S.pcg(A, S.to_dev(b), P, tol=1e-12)
    assert full.flag == 0 and cold.flag == 0 and full.res0 != cold.res0
    # each within cond(A) * tol = 160 * 1e-12 (relative to the start residual) of the solution
    assert float((full.x - cold.x).norm()) <= 2e-9 * float(cold.x.norm())
    stopped = S.pcg(A, S.to_dev(b), P, tol=1e-12, maxit=5)
    assert (stopped.flag, stopped.iterations) == (1, 6)
    zero = S.pcg(A, S.to_dev(np.zeros(Ah.n)), P, tol=1e-12)
    assert (zero.flag, zero.iterations) == (0, 0) and not zero.x.any()
    bad = b.copy()
    bad[17] = np.nan
    assert S.pcg(A, S.to_dev(bad), P, tol=1e-12).flag == 2


def test_solve_longer_than_one_launch():
    """A path of 12000 nodes takes about as many iterations: 9001 of them are
    one launch of 8192 and the rest.  The recurrence's residual is the true one
    to rounding (1e-16 per iteration, relative to the largest residual) if and
    only if the second launch went on from the first one's x, r and p."""
    Ah = grid_laplacian([12000], 1e-9)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    b = S.to_dev(np.random.default_rng(9).standard_normal(Ah.n))
    res = S.pcg(A, b, P, tol=0.0, maxit=9000)
    assert (res.flag, res.iterations) == (1, 9001)
    assert len(res.history) == 9002 and np.isfinite(res.history).all()
    assert abs(res.true_res - res.history[-1]) <= 9001 * 1e-16 * 100 * res.history.max()
    first = S.pcg(A, b, P, tol=0.0, maxit=8300)
    assert np.array_equal(res.history[:8302], first.history)


def test_batch_of_uneven_systems_equals_single_solves():
    """One launch over systems of one row to several workgroups: each system's
    team has the workgroups its own solve would have, so x, iteration count
    and flag are the single solves' bit for bit, whatever shares the launch."""
    dims = [[1], [2048], [64, 32], [2049], [7, 9], [70, 90], [3], [130, 101], [61, 67]]
    dims += [[5, 5 + k % 7] for k in range(300)]  # more teams than the chip has CUs
    systems = [grid_laplacian(d, 0.05) for d in dims]
    rng = np.random.default_rng(11)
    rhs = [rng.standard_normal(A.n) for A in systems]
    rhs[4][:] = 0.0
    B = S.Batch.from_systems(systems, rhs)
    x, it, fl, r0, rs, _ = S.pcg_batched(B, tol=1e-10, block=-1)
    again, *_ = S.pcg_batched(B, tol=1e-10, block=-1)
    assert torch.equal(x, again)
    for k in list(range(9)) + [9, 100, 308]:
        A = S.DeviceCSR.from_csr(systems[k])
        P = S.make_preconditioner(A, systems[k], "line_jacobi")
        one = S.pcg(A, S.to_dev(rhs[k]), P, tol=1e-10)
        assert (it[k], fl[k], r0[k]) == (one.iterations, one.flag, one.res0), k
        assert torch.equal(B.split(x)[k], one.x), k
    assert it[4] == 0 and fl[4] == 0
