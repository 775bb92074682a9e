"""A one-launch Jacobi solve whose workgroups wait too long for each other (they
may not all be running, where something else holds a part of the GPU) goes by
launches, from the start vector, without an error.  Forced here by letting a
wait look twice only: x, iterations and residuals are then those of
resident_polls 0, which takes the launches at once, bit for bit."""
import numpy as np
import pytest
import torch

from lap_amd import lib as L
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian

pytestmark = pytest.mark.gpu


@pytest.fixture
def polls():
    start = S.set_option("resident_polls", 0)
    yield lambda v: S.set_option("resident_polls", v)
    S.set_option("resident_polls", start)


def test_option_range():
    start = S.set_option("resident_polls", 0)
    assert start == 1 << 23
    assert S.set_option("resident_polls", -1) == 0 and L.load().lap_last_status() != 0
    L.load().lap_clear_error()
    assert S.set_option("resident_polls", 1 << 30) == 0
    assert S.set_option("resident_polls", start) == 1 << 30
    assert L.load().lap_last_status() == 0


@pytest.mark.parametrize("dims", [[130, 90], [23, 24, 25], [512, 512]])
def test_single_solve(dims, polls):
    Ah = grid_laplacian(dims, 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    rng = np.random.default_rng(5)
    b, x0 = S.to_dev(rng.standard_normal(Ah.n)), S.to_dev(rng.standard_normal(Ah.n))
    launches = S.pcg(A, b, P, tol=1e-10, x0=x0)
    polls(1 << 23)
    resident = S.pcg(A, b, P, tol=1e-10, x0=x0)
    assert not np.array_equal(resident.history, launches.history)  # (two orders of the sums)
    polls(1)
    cut = S.pcg(A, b, P, tol=1e-10, x0=x0)
    assert L.load().lap_last_status() == 0
    assert (cut.iterations, cut.flag) == (launches.iterations, 0)
    assert torch.equal(cut.x, launches.x) and np.array_equal(cut.history, launches.history)
    polls(1 << 23)
    again = S.pcg(A, b, P, tol=1e-10, x0=x0)
    assert torch.equal(again.x, resident.x) and np.array_equal(again.history, resident.history)


def test_batch(polls):
    systems = [grid_laplacian(d, 0.05) for d in ([130, 101], [7, 9], [70, 90], [2048], [3])]
    rng = np.random.default_rng(6)
    B = S.Batch.from_systems(systems, [rng.standard_normal(A.n) for A in systems])
    x0 = S.to_dev(rng.standard_normal(B.A.n))
    launches = S.pcg_batched(B, tol=1e-10, block=-1, x0=x0)
    polls(1 << 23)
    resident = S.pcg_batched(B, tol=1e-10, block=-1, x0=x0)
    polls(1)
    cut = S.pcg_batched(B, tol=1e-10, block=-1, x0=x0)
    assert torch.equal(cut[0], launches[0]) and not torch.equal(cut[0], resident[0])
    for k in range(1, 5):
        assert np.array_equal(cut[k], launches[k]), k
