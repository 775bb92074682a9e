"""One-launch Jacobi solves at their limits: 2^18 rows of 9 entries (a row per
thread) and one more, 2^19 rows of up to 8 and one more, which goes by launches.
Twelve iterations against the oracle's: the dot products are summed in other
orders (relative 1e-16 per iteration, amplified by the residual's reduction, at
most 1e3); 1e-10 leaves three digits."""
import numpy as np
import pytest

from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_rewritten_columns import circulant

pytestmark = pytest.mark.gpu

CASES = {
    "2^18 rows of 9": (lambda: circulant(1 << 18, [1, 2, 500, 501], 1), True),
    "2^18 + 1 rows of 9": (lambda: circulant((1 << 18) + 1, [1, 2, 500, 501], 1), False),
    "2^19 rows of 7": (lambda: circulant(1 << 19, [1, 64, 500], 1), True),
    "2^19 + 1 rows of 7": (lambda: circulant((1 << 19) + 1, [1, 64, 500], 1), False),
    "2^19 rows of 5": (lambda: grid_laplacian([1024, 512], 0.05), True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_last_that_fits_and_first_that_does_not(orc, name):
    make, one_launch = CASES[name]
    Ah = make()
    b = np.random.default_rng(28).standard_normal(Ah.n)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    res = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=11)
    xo, ito, flo, _ = orc.cg(Ah, b, "line_jacobi", tol=0.0, maxit=11)
    assert (res.iterations, res.flag) == (ito, flo)
    x = res.x.cpu().numpy()
    assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)
    start = S.set_option("resident_polls", 0)
    try:
        launches = S.pcg(A, S.to_dev(b), P, tol=0.0, maxit=11)
    finally:
        S.set_option("resident_polls", start)
    assert np.array_equal(launches.history, res.history) == (not one_launch)
