"""Sweeps of triangles of which a few rows are much longer than the rest (rows
that wrap round), so that their tables are 8 or 16 wide: sweeps of L and U together
keep the CSR arrays at 16, single sweeps take row classes.  Bitwise the CSR solve."""
import numpy as np
import pytest

from lap_amd.problems import CSR
from test_gpu_cls import MIN_ROWS, both, same

import torch  # noqa: F401  (the solves' device)

pytestmark = pytest.mark.gpu


def ring(n, m):
    """i connected to i +- 1 .. m around a ring: 2 m + 1 entries in every row."""
    off = np.concatenate([np.arange(-m, 0), np.arange(0, m + 1)])
    ja = (np.arange(n)[:, None] + off[None, :]) % n
    a = np.where(off == 0, 2.0 * m + 0.05, -1.0)[None, :].repeat(n, 0)
    order = np.argsort(ja, axis=1)
    return CSR(n, (np.arange(n + 1) * (2 * m + 1)).astype(np.int32),
               np.take_along_axis(ja, order, 1).reshape(-1).astype(np.int32),
               np.take_along_axis(a, order, 1).reshape(-1))


@pytest.mark.parametrize("m", [4, 5, 6, 7])
@pytest.mark.parametrize("kind,mk", [("it_jacobi", (1, 2)), ("GS_it2", (1, 2)), ("GS_it", (2, 1))])
def test_ring(m, kind, mk):
    Ah = ring(MIN_ROWS + 3, m)
    b = np.random.default_rng(24).standard_normal(Ah.n)
    same(*both(Ah, kind, b, maxit=20, mk=mk))
