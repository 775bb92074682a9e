"""lap_pcg_spmv_timed runs the SpMV that a solve of the matrix runs: over row
classes for large systems with few distinct rows, with the CSR values otherwise.
The product is hip_csr_matvec's bit for bit."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_cls import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["first_encoded", "last_csr", "cube_odd", "row_15", "row_17",
                                  "too_many"])
def test_product(name):
    A = S.DeviceCSR.from_csr(CASES[name]())
    x = S.to_dev(np.random.default_rng(29).standard_normal(A.n))
    y = torch.zeros_like(x)
    assert S.spmv_timed(A, x, y, 2, fused=True) > 0
    assert torch.equal(y, S.spmv(A, x))


def test_a_large_grid_is_read_as_classes():
    """A byte a row instead of 84: half the time or less (118 and 352 us at 256^3)."""
    Ah = grid_laplacian([200, 200, 200], 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    B = S.DeviceCSR(A.n, A.ia, A.ja, A.a * torch.linspace(1.0, 2.0, A.nnz, dtype=torch.float64,
                                                          device=S.DEV))
    B.forget()
    x = S.to_dev(np.random.default_rng(30).standard_normal(A.n))
    y = torch.zeros_like(x)
    ms = [min(S.spmv_timed(M, x, y, 50, fused=True) for _ in range(3)) for M in (A, B)]
    print(f"[diag] classes {ms[0] * 1e3:.1f} us, CSR {ms[1] * 1e3:.1f} us", flush=True)
    assert ms[0] < 0.8 * ms[1]
