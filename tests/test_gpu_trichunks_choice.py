"""Triangles whose chunks and level launches are timed against each other, or
that have few levels: the chunks (sptrsv_mode 4), the faster of the two (3) and
the level launches (0) give the same bits, in single solves through IC0, whole
GS_std and IC0 PCG runs and the mixed-precision IC0 solve."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import CSR, from_coo, grid_laplacian
from test_gpu_rewritten_columns import circulant
from test_gpu_trichunks import _long_range

pytestmark = pytest.mark.gpu


def shuffled(A):
    p = np.random.default_rng(1).permutation(A.n)
    r = np.repeat(np.arange(A.n), np.diff(A.ia))
    k = A.ja <= r
    a, b = p[r[k]], p[A.ja[k]]
    return from_coo(A.n, np.maximum(a, b), np.minimum(a, b), A.a[k], symmetric=True)


CASES = {
    "diagonal": lambda: CSR(3000, np.arange(3001, dtype=np.int32), np.arange(3000, dtype=np.int32),
                            1.0 + np.arange(3000) % 5),
    "line_of_3": lambda: grid_laplacian([3], 0.1),
    "line_of_4": lambda: grid_laplacian([4], 0.1),
    "shuffled_plane": lambda: shuffled(grid_laplacian([100, 90], 0.05)),
    "shuffled_line": lambda: shuffled(grid_laplacian([30011], 0.05)),
    "far_circulant": lambda: circulant(50000, [2300, 7000], 1),
    "long_range": lambda: _long_range(20011),
}


def runs(Ah, mode):
    A = S.DeviceCSR.from_csr(Ah)
    b = S.to_dev(np.random.default_rng(23).standard_normal(Ah.n))
    old = S.set_option("sptrsv_mode", mode)
    try:
        P = S.make_preconditioner(A, Ah, "ichol")
        G = S.make_preconditioner(A, Ah, "GS_std")
        out = [S.prec_apply(A, P, b)]
        for r in (S.pcg(A, b, P, tol=1e-8, maxit=40), S.pcg(A, b, G, tol=1e-8, maxit=40),
                  S.pcg_mixed(A, b, P, tol=1e-8, maxit=40)):
            out += [r.x, torch.from_numpy(r.history)]
        return out
    finally:
        S.set_option("sptrsv_mode", old)


@pytest.mark.parametrize("name", list(CASES))
def test_every_mode_gives_the_same_bits(name):
    Ah = CASES[name]()
    levels = runs(Ah, 0)
    for mode in (4, 3, 3):
        for got, want in zip(runs(Ah, mode), levels):
            assert torch.equal(got, want), mode
