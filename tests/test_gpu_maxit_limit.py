"""maxit = 2^31 - 1 is a limit like any other: single solves and batches, in one
launch and by launches, block and mixed-precision solves stop where they do with
a smaller one."""
import ctypes as C

import numpy as np
import pytest
import torch

from lap_amd import lib as L
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian

pytestmark = pytest.mark.gpu

MOST = 2**31 - 1


@pytest.fixture(params=[0, 1 << 23], ids=["launches", "one_launch"])
def route(request):
    start = S.set_option("resident_polls", request.param)
    yield
    S.set_option("resident_polls", start)
    L.load().lap_release_all()  # (a device history of 17 GB)


def test_single_solves(route):
    Ah = grid_laplacian([70, 60], 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    b = S.to_dev(np.random.default_rng(21).standard_normal(Ah.n))
    want = S.pcg(A, b, P, tol=1e-10)
    wantm = S.pcg_mixed(A, b, P, tol=1e-10)
    args = [S.ptr(v) for v in (A.ia, A.ja, A.a)]
    x, info = torch.zeros_like(b), L.SolveInfo()
    torch.cuda.synchronize()
    assert L.load().lap_pcg(A.n, A.nnz, *args, S.ptr(x), S.ptr(b), 1e-10, C.byref(P.pdata), MOST,
                            None, C.byref(info)) == 0
    assert (info.iterations, info.flag) == (want.iterations, 0) and torch.equal(x, want.x)
    x.zero_()
    torch.cuda.synchronize()
    assert L.load().lap_pcg_mixed(A.n, A.nnz, *args, S.ptr(x), S.ptr(b), 1e-10, C.byref(P.pdata),
                                  MOST, 0.01, None, C.byref(info)) == 0
    assert (info.iterations, info.flag) == (wantm.iterations, 0) and torch.equal(x, wantm.x)


def test_batch_and_block(route):
    systems = [grid_laplacian(d, 0.05) for d in ([70, 60], [9, 11], [130, 101])]
    rng = np.random.default_rng(22)
    B = S.Batch.from_systems(systems, [rng.standard_normal(A.n) for A in systems])
    want = S.pcg_batched(B, tol=1e-10, block=-1)
    got = S.pcg_batched(B, tol=1e-10, block=-1, maxit=MOST)
    assert torch.equal(got[0], want[0]) and not got[2].any() and np.array_equal(got[1], want[1])
    R = torch.randn(B.A.n, 4, dtype=torch.float64, device=S.DEV)
    wb = S.pcg_block(B.A, R, B.d_r, tol=1e-10)
    gb = S.pcg_block(B.A, R, B.d_r, tol=1e-10, maxit=MOST)
    assert torch.equal(gb.x, wb.x) and np.array_equal(gb.iterations, wb.iterations)
