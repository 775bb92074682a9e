"""Device memory and the one-launch Jacobi solve: while there is too little for
its plan the solve goes by launches, and afterwards it is the one launch again;
plans take what their halos need, and those that do not fit take nothing."""
from contextlib import contextmanager

import numpy as np
import pytest
import torch

from lap_amd import lib as L
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_rewritten_columns import circulant

pytestmark = pytest.mark.gpu

MB = 1 << 20


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@contextmanager
def memory_left(n):
    """All but n bytes of the device's memory taken."""
    torch.cuda.empty_cache()
    held, size = [], 1 << 36
    while size >= 4 * MB:
        if free_bytes() - n > size:
            held.append(torch.empty(size, dtype=torch.uint8, device=S.DEV))
        else:
            size //= 2
    try:
        yield
    finally:
        held.clear()
        torch.cuda.empty_cache()


def by_launches(A, P, b):
    """The history by launches (its sums differ from one launch's in the last bits)."""
    start = S.set_option("resident_polls", 0)
    launches = S.pcg(A, b, P, tol=1e-10)
    S.set_option("resident_polls", start)
    return launches.history


def test_short_of_memory_for_a_while():
    Ah = grid_laplacian([300, 200], 0.05)
    A, other = S.DeviceCSR.from_csr(Ah), S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    b = S.to_dev(np.random.default_rng(14).standard_normal(Ah.n))
    launches = by_launches(A, P, b)
    resident = S.pcg(other, b, P, tol=1e-10).history
    assert not np.array_equal(launches, resident)
    with memory_left(40 * MB):
        short = S.pcg(A, b, P, tol=1e-10)
        assert L.load().lap_last_status() == 0
    assert np.array_equal(short.history, launches)
    assert np.array_equal(S.pcg(A, b, P, tol=1e-10).history, resident)


def test_batch_short_of_memory_for_a_while():
    rng = np.random.default_rng(15)
    systems = [grid_laplacian([130, 90 + k], 0.05) for k in range(9)]
    B = S.Batch.from_systems(systems, [rng.standard_normal(A.n) for A in systems])
    start = S.set_option("resident_polls", 0)
    launches = S.pcg_batched(B, tol=1e-10, block=-1)
    S.set_option("resident_polls", start)
    with memory_left(40 * MB):
        short = S.pcg_batched(B, tol=1e-10, block=-1)
    assert torch.equal(short[0], launches[0])
    assert not torch.equal(S.pcg_batched(B, tol=1e-10, block=-1)[0], launches[0])


def used_by(solve):
    """What `solve` keeps of the device's memory beyond the first call of its like."""
    solve(0)
    before = free_bytes()
    solve(1)
    return before - free_bytes()


def test_plan_that_does_not_fit_keeps_nothing():
    """150,000 rows whose 16 neighbours are far apart: halos of 16,384 rows."""
    rng = np.random.default_rng(16)
    Ah = circulant(150000, range(5000, 45000, 5000), 1)
    mats = [S.DeviceCSR.from_csr(Ah), S.DeviceCSR.from_csr(Ah)]
    P = S.make_preconditioner(mats[0], Ah, "line_jacobi")
    b = S.to_dev(rng.standard_normal(Ah.n))
    S.pcg(mats[0], b, P, tol=1e-6)
    # (the SpMV plan's row blocks are what is left; the lists alone would be 4.8 MB)
    assert used_by(lambda k: S.pcg(mats[k], b, P, tol=1e-6)) <= 2 * MB


def test_lists_are_as_long_as_the_halos():
    """2000 systems of one workgroup and no halo: 64 MB were 32 KB each."""
    rng = np.random.default_rng(17)
    systems = [grid_laplacian([20, 20], 0.05)] * 2000
    rhs = [rng.standard_normal(400) for _ in systems]
    batches = [S.Batch.from_systems(systems, rhs) for _ in range(2)]
    S.pcg_batched(batches[0], tol=1e-6, block=-1)
    # boxes 13 + 2000 * 0.4, slots 2 * 3.9, marks 0.8 MB, and 2 MB steps of each
    assert used_by(lambda k: S.pcg_batched(batches[k], tol=1e-6, block=-1)) <= 32 * MB
