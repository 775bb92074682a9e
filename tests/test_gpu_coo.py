"""COO -> CSR on the device at the sizes where its kernels change course: rows
of 32, 33, 4096 and 4097 entries, 128 rows with 2048 entries and one more,
runs of one row across waves and workgroups, every order of the entries,
repeated entries, rectangular and symmetric.  The expected arrays are a stable
sort by (row, column) of the entries with each mirror after its entry; all
values are compared exactly."""
import numpy as np
import pytest
import torch

from lap_amd import io as IO
from lap_amd import solver as S

pytestmark = pytest.mark.gpu


def expected(n, r, c, v, sym):
    if sym:
        off = r != c
        seq = np.concatenate([2 * np.arange(len(r)), 2 * np.nonzero(off)[0] + 1])
        r, c, v = (np.concatenate([r, c[off]]), np.concatenate([c, r[off]]),
                   np.concatenate([v, v[off]]))
    else:
        seq = np.arange(len(r))
    order = np.lexsort((seq, c, r))
    ia = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    return ia, c[order], v[order]


def check(n, r, c, sym, m=None, seed=0):
    v = np.random.default_rng(seed).standard_normal(len(r))
    rd, cd = (torch.from_numpy(x.astype(np.int32)).to(S.DEV) for x in (r, c))
    A = IO.coo_to_csr(n, rd, cd, S.to_dev(v), sym, m)
    ia, ja, a = expected(n, r, c, v, sym)
    assert np.array_equal(A.ia.cpu().numpy(), ia)
    assert np.array_equal(A.ja.cpu().numpy(), ja)
    assert np.array_equal(A.a.cpu().numpy().view(np.int64), a.view(np.int64))


def orders(r, c):
    rng = np.random.default_rng(1)
    yield np.arange(len(r))
    yield np.lexsort((r, c))
    yield np.lexsort((c, r))[::-1]
    yield rng.permutation(len(r))


@pytest.mark.parametrize("lengths", [[1], [32] * 5, [33, 1, 32], [16] * 128, [16] * 127 + [17],
                                     [16] * 300 + [17] * 300, [0, 0, 3, 0], [2] * 129, [4096, 5],
                                     [4097, 32, 33], [31, 5000, 0, 9000, 7]])
def test_row_lengths(lengths):
    rng = np.random.default_rng(len(lengths))
    m = max(lengths) + 3
    r = np.repeat(np.arange(len(lengths)), lengths)
    c = np.concatenate([rng.permutation(m)[:k] for k in lengths])
    for o in orders(r, c):
        check(len(lengths), r[o], c[o], False, m)


@pytest.mark.parametrize("n,nnz", [(1, 1), (7, 63), (50, 64), (50, 65), (300, 1000), (5000, 30001),
                                   (40, 70000)])
def test_symmetric_with_repeats(n, nnz):
    rng = np.random.default_rng(nnz)
    r, c = rng.integers(0, n, nnz), rng.integers(0, n, nnz)
    for o in orders(r, c):
        check(n, r[o], c[o], True, seed=n)


def test_runs_across_workgroups():
    """One column's entries fill several workgroups; so do a row's."""
    n = 2000
    r = np.concatenate([np.arange(n), np.full(1500, 17), np.arange(n)])
    c = np.concatenate([np.full(n, 5), np.arange(1500), np.arange(n)])
    check(n, r, c, True)
    check(n, r, c, False)
