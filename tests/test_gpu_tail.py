"""PCG with IC0 and GS_std where the triangular solve's copy back, the update of w
and the dot product r.w are one pass (chunked solves) against the separate
launches (level solves): the same values in the same order, so bit for bit equal.
One row block to more of them than workgroups, one and two sweeps."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import grid_laplacian

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [[5], [255], [17, 16], [64, 33], [31, 29, 33], [83, 81, 79]])
@pytest.mark.parametrize("kind,k", [("ichol", 1), ("GS_std", 1), ("GS_std", 2)])
def test_tail_is_bitwise_the_separate_launches(dims, kind, k):
    Ah = grid_laplacian(dims, 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    b = S.to_dev(np.random.default_rng(5).standard_normal(Ah.n))
    out = []
    for mode in (3, 0):
        old = S.set_option("sptrsv_mode", mode)
        try:
            P = S.make_preconditioner(A, Ah, kind, 1, k)
            out.append(S.pcg(A, b, P, tol=0.0, maxit=12))
        finally:
            S.set_option("sptrsv_mode", old)
    r, s = out
    assert (r.iterations, r.flag) == (s.iterations, s.flag)
    assert np.array_equal(r.history, s.history, equal_nan=True)
    assert torch.equal(r.x.view(torch.int64), s.x.view(torch.int64))
