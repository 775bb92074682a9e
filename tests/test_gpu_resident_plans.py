"""Several plans of one-launch Jacobi solves kept at once: a matrix whose halo
needs most of the LDS, one of the same kernel with next to none, and the first
one again; single solves and batches.  The repeated result is the first one."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_rewritten_columns import circulant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide,narrow", [
    (lambda: circulant(40000, [5000, 11000], 1), lambda: grid_laplacian([64, 64], 0.05)),
    (lambda: circulant(40000, [1, 3, 5000, 17000], 1), lambda: circulant(3000, range(1, 5), 2)),
    (lambda: circulant(20000, [3, 1200, 2400, 3600, 4800, 6000], 1),
     lambda: circulant(3000, range(1, 7), 2)),
])
def test_single_solves(wide, narrow):
    runs = []
    for h in (wide(), narrow()):
        A = S.DeviceCSR.from_csr(h)
        b = S.to_dev(np.random.default_rng(h.n).standard_normal(h.n))
        runs.append((A, b, S.make_preconditioner(A, h, "line_jacobi")))
    first = [S.pcg(*r, tol=1e-10) for r in runs]
    again = [S.pcg(*r, tol=1e-10) for r in runs]
    for f, g in zip(first, again):
        assert f.flag == 0 and torch.equal(f.x, g.x) and np.array_equal(f.history, g.history)


def test_batches():
    rng = np.random.default_rng(13)
    batches = []
    for systems in ([circulant(40000, [5000, 11000], k) for k in range(25)],
                    [grid_laplacian([41, 60], 0.05)] * 500):
        batches.append(S.Batch.from_systems(systems, [rng.standard_normal(A.n) for A in systems]))
    first = [S.pcg_batched(B, tol=1e-10, block=-1) for B in batches]
    again = [S.pcg_batched(B, tol=1e-10, block=-1) for B in batches]
    for f, g in zip(first, again):
        assert not f[2].any() and torch.equal(f[0], g[0]) and np.array_equal(f[1], g[1])
