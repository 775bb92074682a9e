"""The SpMM where rows are long or few (k >= 16): a row per lane group up to
16,384 rows and for rows of more than 256 entries, chunks of 16 rows beyond, whose
nonzeros fit the LDS or are read in windows.  Every column is the CSR sum bit for
bit; block solves equal those of fewer columns, which never take these routes."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import CSR, grid_laplacian
from test_gpu_spmm_chunks import rows_of

pytestmark = pytest.mark.gpu


def lengths(n, kind):
    i = np.arange(n)
    few = (i % 7) % 4
    return {"16": 16 + 0 * i,                                # 256 of 256 in 16 rows
            "spills": 16 + (i % 32 == 7),                    # 257 in every other 16 rows
            "empty": (i % 5 == 2) * 4,
            "to_256": np.where(i % 97 == 5, 256, few),       # a window and no more
            "uneven": np.where(i % 16 < 2, 130 + i % 120, few),  # some groups end early
            "to_257": np.where(i == n // 2, 257, few),       # a row per group
            "hubs": np.where(i < 5, 3000 + 17 * i, few)}[kind]


@pytest.mark.parametrize("k", [16, 32, 64])
@pytest.mark.parametrize("n,kind", [(16385, "16"), (16385, "spills"), (16400, "empty"),
                                    (16385, "to_256"), (16391, "uneven"), (16385, "to_257"),
                                    (20000, "hubs"), (16384, "uneven"), (4000, "hubs"),
                                    (259, "to_256"), (260, "to_257")])
def test_rows(orc, n, kind, k):
    Ah = rows_of(lengths(n, kind), seed=n)
    A = S.DeviceCSR.from_csr(Ah)
    X = np.random.default_rng(k).standard_normal((n, k))
    want = np.stack([orc.matvec(Ah, X[:, j].copy()) for j in range(k)], axis=1)
    for tile in (1, 2, 4):
        assert np.array_equal(S.spmm(A, S.to_dev(X), tile=tile).cpu().numpy(), want), tile


@pytest.mark.parametrize("n,kind", [(16385, "uneven"), (4000, "hubs")])
def test_not_finite(orc, n, kind):
    Ah = rows_of(lengths(n, kind), seed=n)
    A = S.DeviceCSR.from_csr(Ah)
    X = np.random.default_rng(1).standard_normal((n, 64))
    X[0, 0], X[500, 33], X[-1, 63] = np.inf, np.nan, -np.inf
    with np.errstate(invalid="ignore"):
        want = np.stack([orc.matvec(Ah, X[:, j].copy()) for j in range(64)], axis=1)
    assert np.array_equal(S.spmm(A, S.to_dev(X)).cpu().numpy(), want, equal_nan=True)


def test_hub_in_an_operand_past_4_gb():
    n, k = (1 << 23) + 77, 64
    ja = np.minimum(np.arange(n) + 70000, n - 1)
    hub = np.linspace(0, n - 1, 300).astype(np.int64)
    ia = np.arange(n + 1, dtype=np.int64)
    ia[1:] += 299  # row 0 is the hub
    Ah = CSR(n, ia.astype(np.int32), np.concatenate([hub, ja[1:]]).astype(np.int32),
             1.0 + (np.arange(n + 299) % 11) / 7.0)
    A = S.DeviceCSR.from_csr(Ah)
    X = torch.randn(n, k, dtype=torch.float64, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(3))
    Y = S.spmm(A, X)
    for j in (0, 63):
        assert torch.equal(Y[:, j], S.spmv(A, X[:, j].contiguous()))


@pytest.mark.parametrize("dims", [[30, 29, 28], [20, 20, 20]])  # chunks, a row per group
@pytest.mark.parametrize("k", [16, 32, 64])
def test_block_solve(dims, k):
    """Twelve iterations; the dot products of the two are summed in different
    orders (1e-16 per iteration, amplified by the residual's reduction, at most
    1e3): 1e-10 leaves three digits."""
    Ah = grid_laplacian(dims, 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "line_jacobi")
    d_r = P.keep["d_r"]
    B = S.to_dev(np.random.default_rng(k).standard_normal((Ah.n, k)))
    X0 = S.to_dev(np.random.default_rng(k + 1).standard_normal((Ah.n, k)))
    got = S.pcg_block(A, B, d_r, tol=0.0, maxit=11, x0=X0)
    assert (got.iterations == 12).all()
    for j in (0, 8, k - 8):
        want = S.pcg_block(A, B[:, j:j + 8].contiguous(), d_r, tol=0.0, maxit=11,
                           x0=X0[:, j:j + 8].contiguous())
        assert float((got.x[:, j:j + 8] - want.x).norm()) <= 1e-10 * float(want.x.norm()), j
        assert np.allclose(got.res[j:j + 8], want.res, rtol=1e-10, atol=0)
