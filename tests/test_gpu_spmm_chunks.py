"""SpMM by chunks of rows (lap_csr_matmat, lap_pcg_block): every column is the
CSR sum bit for bit.  Sizes around a chunk and a workgroup, chunks whose
nonzeros just fit, just do not, and lie in one row, empty rows, infinities,
row blocks dealt to the XCDs in groups, and a right operand past 4 GB."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import CSR, grid_laplacian

pytestmark = pytest.mark.gpu


def rows_of(lengths, seed=0):
    """A matrix with rows of these lengths at random ascending columns."""
    n = len(lengths)
    rng = np.random.default_rng(seed)
    ia = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ja = np.concatenate([np.sort(rng.choice(n, m, replace=False)) for m in lengths]
                        + [np.zeros(0, np.int64)])
    return CSR(n, ia, ja.astype(np.int32), rng.standard_normal(ia[-1]))


def lengths(n, kind):
    i = np.arange(n)
    return {"3": np.minimum(3, n) + 0 * i,
            "empty": (i % 5 == 2) * np.minimum(4, n),
            "fits": np.minimum(n, 16) + 0 * i,            # 256 of 256 in 16 rows
            "spills": np.minimum(n, 16) + (i % 32 == 7),  # 257 in every other 16 rows
            "wide_fits": np.minimum(n, 8) + 0 * i,        # 512 of 512 in 64 rows
            "wide_spills": np.minimum(n, 8) + (i % 64 == 7),
            "one_row": np.where(i == n // 2, min(n, 300), 1)}[kind]


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("n,kind", [(1, "3"), (15, "3"), (16, "empty"), (17, "3"), (63, "empty"),
                                    (64, "3"), (65, "3"), (257, "empty"), (1000, "fits"),
                                    (1000, "spills"), (1000, "wide_fits"), (1000, "wide_spills"),
                                    (1000, "one_row")])
def test_chunks(orc, n, kind, k):
    Ah = rows_of(lengths(n, kind))
    A = S.DeviceCSR.from_csr(Ah)
    X = np.random.default_rng(k).standard_normal((n, k))
    want = np.stack([orc.matvec(Ah, X[:, j].copy()) for j in range(k)], axis=1)
    for tile in (1, 2, 4):
        assert np.array_equal(S.spmm(A, S.to_dev(X), tile=tile).cpu().numpy(), want), tile


@pytest.mark.parametrize("dims", [[40, 37, 33], [257, 190], [31, 8, 200]])
@pytest.mark.parametrize("k,per_cu", [(32, 4), (8, 4), (16, 1), (2, 16)])
def test_groups(orc, dims, k, per_cu):
    Ah = grid_laplacian(dims, 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    X = np.random.default_rng(k).standard_normal((Ah.n, k))
    want = np.stack([orc.matvec(Ah, X[:, j].copy()) for j in range(k)], axis=1)
    old = S.set_option("spmm_wg_per_cu", per_cu)
    try:
        assert np.array_equal(S.spmm(A, S.to_dev(X)).cpu().numpy(), want)
    finally:
        S.set_option("spmm_wg_per_cu", old)


def test_not_finite(orc):
    Ah = grid_laplacian([40, 30], 0.05)
    A = S.DeviceCSR.from_csr(Ah)
    X = np.random.default_rng(1).standard_normal((Ah.n, 8))
    X[0, 0], X[500, 3], X[-1, 7] = np.inf, np.nan, -np.inf
    with np.errstate(invalid="ignore"):
        want = np.stack([orc.matvec(Ah, X[:, j].copy()) for j in range(8)], axis=1)
    assert np.array_equal(S.spmm(A, S.to_dev(X)).cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("n", [(1 << 22) + (1 << 20), (1 << 23) - 1, (1 << 23) + 77])
def test_operand_around_4_gb(n):
    """2.7 GB, the last size within 32-bit offsets, and past it."""
    k = 64
    i = np.arange(n, dtype=np.int64)
    ja = np.stack([np.maximum(i - 5, 0), i, np.minimum(i + 70000, n - 1)], axis=1)
    ja[:, 1] = np.where(ja[:, 0] == ja[:, 1], ja[:, 0], ja[:, 1])
    Ah = CSR(n, (3 * np.arange(n + 1)).astype(np.int32), ja.reshape(-1).astype(np.int32),
             1.0 + (np.arange(3 * n) % 11) / 7.0)
    A = S.DeviceCSR.from_csr(Ah)
    X = torch.randn(n, k, dtype=torch.float64, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(2))
    Y = S.spmm(A, X, tile=2)
    for j in (0, 63):
        assert torch.equal(Y[:, j], S.spmv(A, X[:, j].contiguous()))
