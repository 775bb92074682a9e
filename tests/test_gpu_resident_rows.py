"""The resident solve of short rows: one to 240 workgroups, rows of 5 entries and
more, and batches on either side of the rule for two workgroups per CU.

Compared with the oracle after exactly as many iterations, as the smaller
workgroups are: the dot products are summed in another order, relative 1e-16 per
iteration amplified by at most 1e3; 1e-10 leaves three digits."""
import numpy as np
import pytest
import torch

import oracle
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_resident import circulant

pytestmark = pytest.mark.gpu

CASES = {
    "line_2048": lambda: grid_laplacian([2048], 0.05),
    "line_2049": lambda: grid_laplacian([2049], 0.05),
    "plane_64x64": lambda: grid_laplacian([64, 64], 0.05),  # 4096: one workgroup
    "line_4097": lambda: grid_laplacian([4097], 0.05),
    "plane_255x257": lambda: grid_laplacian([255, 257], 0.05),  # 65535
    "plane_256x256": lambda: grid_laplacian([256, 256], 0.05),
    "circulant_5": lambda: circulant(70001, [1, 300]),
    "circulant_5_far": lambda: circulant(65537, [1, 30000]),
    "circulant_7": lambda: circulant(65537, [1, 2, 300]),
    "plane_700x701": lambda: grid_laplacian([700, 701], 0.05),
}


@pytest.mark.parametrize("name", list(CASES))
def test_fixed_iterations_match_the_oracle(name):
    Ah = CASES[name]()
    b = np.random.default_rng(7).standard_normal(Ah.n)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    res = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=11)
    xo, ito, flo, _ = oracle.Oracle().cg(Ah, b, "line_jacobi", tol=0.0, maxit=11)
    assert (res.iterations, res.flag) == (ito, flo)
    x = res.x.cpu().numpy()
    assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)
    again = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=11)
    assert torch.equal(again.x, res.x) and np.array_equal(again.history, res.history)


@pytest.mark.parametrize("systems", [300, 500])
def test_batch_equals_single_solves(systems):
    """Systems of 1 to 5 x 1024 rows in one launch, of 512 threads per workgroup
    for 500 of them and 1024 for 300 and each alone: the same bits."""
    rng = np.random.default_rng(1)
    dims = [(1, 1), (64, 64), (2048, 1)] + [tuple(map(int, rng.integers(20, 72, 2)))
                                            for _ in range(systems - 3)]
    mats = [grid_laplacian(list(d), 0.05) for d in dims]
    rhs = [rng.standard_normal(A.n) for A in mats]
    B = S.Batch.from_systems(mats, rhs)
    x, it, fl, *_ = S.pcg_batched(B, block=-1, tol=1e-10)
    assert not fl.any()
    for s in [0, 1, 2, 3, 57, 299]:
        A = S.DeviceCSR.from_csr(mats[s])
        P = S.make_preconditioner(A, mats[s], "line_jacobi")
        r = S.pcg(A, S.to_dev(rhs[s]), P, tol=1e-10)
        assert int(it[s]) == r.iterations
        assert torch.equal(B.split(x)[s], r.x)


@pytest.mark.parametrize("systems", [32768, 32769])
def test_batches_around_the_most_workgroups(systems):
    """Past the limit the batch goes by launches: the same solutions (2 x 2 grids,
    exact after 3 iterations)."""
    A1 = grid_laplacian([2, 2], 0.5)
    rng = np.random.default_rng(2)
    rhs = rng.standard_normal((systems, 4))
    B = S.Batch.from_systems([A1] * systems, list(rhs))
    x, it, fl, *_ = S.pcg_batched(B, block=-1, tol=1e-12)
    dense = np.zeros((4, 4))
    for r in range(4):
        dense[r, A1.ja[A1.ia[r]:A1.ia[r + 1]]] = A1.a[A1.ia[r]:A1.ia[r + 1]]
    want = np.linalg.solve(dense, rhs.T).T.ravel()
    assert not fl.any()
    assert np.abs(x.cpu().numpy() - want).max() <= 1e-9 * np.abs(want).max()
