"""A batch of three systems of 100 workgroups each, which do not fit the GPU
together: the third one's first workgroups start beside the other two and wait
for the rest.  The systems take 100,001 iterations each (half a second); the
waits are cut to 600,000 looks (about 0.1 s), which a launch of a limited number
of iterations (0.04 s) stays below.  Each system's result is its single solve's
bit for bit; by launches (a wait that ran out) it would not be."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import grid_laplacian

pytestmark = pytest.mark.gpu


def test_systems_that_wait_for_each_other():
    systems = [grid_laplacian([100 * 2048], 1e-9) for _ in range(3)]
    systems.append(grid_laplacian([70, 60], 0.05))  # ends in the first launch
    rng = np.random.default_rng(12)
    rhs = [rng.standard_normal(A.n) for A in systems]
    tol, maxit = 1e-12, 100000
    one = []
    for Ah, b in zip(systems, rhs):
        A = S.DeviceCSR.from_csr(Ah)
        one.append(S.pcg(A, S.to_dev(b), S.make_preconditioner(A, Ah, "line_jacobi"), tol=tol,
                         maxit=maxit))
    assert [o.flag for o in one] == [1, 1, 1, 0] and one[0].iterations == maxit + 1
    B = S.Batch.from_systems(systems, rhs)
    start = S.set_option("resident_polls", 600000)
    try:
        x, it, fl, r0, rs, ms = S.pcg_batched(B, tol=tol, maxit=maxit, block=-1)
    finally:
        S.set_option("resident_polls", start)
    print(f"[diag] single {one[0].gpu_ms:.0f} ms, batch {ms:.0f} ms", flush=True)
    for k, o in enumerate(one):
        assert (it[k], fl[k], r0[k]) == (o.iterations, o.flag, o.res0), k
        assert torch.equal(B.split(x)[k], o.x), k
