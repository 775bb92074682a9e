"""A chunked triangular solve without the memory for its records goes by levels:
GS_std PCG with all but a little of the device's memory taken, at amounts that
leave room for one triangle's records and for none.  Rows and dot products are
summed in the same order on both routes, so the iterates are equal bit for bit."""
import numpy as np
import pytest
import torch

from lap_amd import lib as L
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_resident_memory import MB, memory_left

pytestmark = pytest.mark.gpu


def test_gs_std_short_of_memory():
    Ah = grid_laplacian([100, 90, 80], 0.05)  # a triangle: 35 MB of rows, 50 MB of records or more
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "GS_std")
    b = S.to_dev(np.random.default_rng(20).standard_normal(Ah.n))
    want = S.pcg(A, b, P, tol=1e-6)
    again = [want]
    for left in (160, 70):
        with memory_left(left * MB):
            got = S.pcg(A, b, P, tol=1e-6)
            assert L.load().lap_last_status() == 0, left
        again.append(got)
        print(f"[diag] {left} MB left: {got.gpu_ms / got.iterations:.2f} ms per iteration", flush=True)
        assert got.flag == 0 and got.iterations == want.iterations, left
        assert torch.equal(got.x, want.x) and np.array_equal(got.history, want.history), left
    assert again[-1].gpu_ms > 2 * want.gpu_ms  # (levels: the last one did run out of memory)
