"""SpMV rows around the lengths where the row sum changes course (24, 40 and 64
entries, a full tile of 2048), and more row blocks than workgroups: every row is
the CSR sum bit for bit; a row past the tile is a tree sum (relative 1e-13: 4096
terms of like size)."""
import numpy as np
import pytest

from lap_amd import solver as S
from lap_amd.problems import CSR

pytestmark = pytest.mark.gpu


def matrix(lengths, n):
    rng = np.random.default_rng(len(lengths))
    ia = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ja = np.concatenate([np.sort(rng.choice(n, m, replace=False)) for m in lengths])
    return CSR(n, ia, ja.astype(np.int32), rng.standard_normal(ia[-1]))


def check(orc, Ah, alpha, beta, exact=slice(None)):
    rng = np.random.default_rng(2)
    x, y = rng.standard_normal(Ah.n), rng.standard_normal(Ah.n)
    got = S.spmv(S.DeviceCSR.from_csr(Ah), S.to_dev(x), S.to_dev(y), alpha, beta).cpu().numpy()
    want = y.copy()
    want = orc.matvec(Ah, x, want, alpha, beta)
    assert np.array_equal(got[exact], want[exact])
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-13 * 4096)


@pytest.mark.parametrize("longest", [23, 24, 39, 40, 56, 63, 64, 65, 255, 1031, 2048, 4096])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.5, 2.0)])
def test_row_lengths(orc, longest, alpha, beta):
    n = 5000
    lengths = np.arange(n) % 7
    lengths[::97] = longest
    lengths[1::97] = max(1, longest - 1)
    check(orc, matrix(lengths, n), alpha, beta, lengths <= 2048)


@pytest.mark.parametrize("n", [2048 * 256, 2048 * 256 + 1, 3 * 2048 * 256 + 77])
@pytest.mark.parametrize("hub", [0, 100])
def test_more_blocks_than_workgroups(orc, n, hub):
    i = np.arange(n)
    ja = np.stack([np.maximum(i - 1, 0), i, np.minimum(i + 1, n - 1)], axis=1)
    keep = np.ones((n, 3), bool)
    keep[0, 0] = keep[-1, 2] = False
    ia = np.concatenate([[0], np.cumsum(keep.sum(1))])
    ja, rows = ja[keep], np.repeat(i, keep.sum(1))
    if hub:  # a row of 100 entries: the deep sum
        ja = np.concatenate([np.arange(hub), ja[ia[1]:]])
        ia = np.concatenate([[0], ia[1:] + hub - ia[1]])
    a = np.random.default_rng(1).standard_normal(len(ja))
    check(orc, CSR(n, ia.astype(np.int32), ja.astype(np.int32), a), 1.0, 0.0)
