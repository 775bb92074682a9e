"""An error of an earlier call, dealt with by its caller, has no part in a later
one-launch Jacobi solve."""
import ctypes as C

import numpy as np
import pytest
import torch

from lap_amd import lib as L
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian

pytestmark = pytest.mark.gpu


def test_solve_after_a_refused_allocation():
    lib = L.load()
    Ah = grid_laplacian([70, 60], 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    b = S.to_dev(np.random.default_rng(18).standard_normal(Ah.n))
    want = S.pcg(A, b, P, tol=1e-10)
    x = torch.zeros_like(b)
    info = L.SolveInfo()
    torch.cuda.synchronize()
    assert lib.mallocForDevice(None, 0x7fffffff, 1 << 20) is None  # 2 PB
    assert lib.lap_last_status() != 0
    lib.lap_clear_error()
    args = [S.ptr(v) for v in (A.ia, A.ja, A.a, x, b)]
    st = lib.lap_pcg(A.n, A.nnz, *args, 1e-10, C.byref(P.pdata), 25000, None, C.byref(info))
    msg = lib.lap_last_error()
    with pytest.raises(RuntimeError, match="out of memory"):  # takes the runtime's last error
        torch.zeros(1000, device=S.DEV).sum()
    assert st == 0, msg
    assert info.iterations == want.iterations and torch.equal(x, want.x)


def test_plan_made_beside_an_error_of_another_call():
    """A recorded error that nobody has cleared yet fails the call's status, as
    ever, but the matrix is solved, and in one launch then and later."""
    lib = L.load()
    Ah = grid_laplacian([70, 60], 0.05)
    A, other = S.DeviceCSR.from_csr(Ah), S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    b = S.to_dev(np.random.default_rng(19).standard_normal(Ah.n))
    want = S.pcg(other, b, P, tol=1e-10)
    x = torch.zeros_like(b)
    info = L.SolveInfo()
    torch.cuda.synchronize()
    assert lib.mallocForDevice(None, 0x7fffffff, 1 << 20) is None
    with pytest.raises(RuntimeError, match="out of memory"):
        torch.zeros(1000, device=S.DEV).sum()
    args = [S.ptr(v) for v in (A.ia, A.ja, A.a, x, b)]
    st = lib.lap_pcg(A.n, A.nnz, *args, 1e-10, C.byref(P.pdata), 25000, None, C.byref(info))
    assert st == lib.lap_last_status() != 0
    lib.lap_clear_error()
    assert info.iterations == want.iterations and torch.equal(x, want.x)
    again = S.pcg(A, b, P, tol=1e-10)
    assert torch.equal(again.x, want.x) and np.array_equal(again.history, want.history)
