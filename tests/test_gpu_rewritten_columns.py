"""A matrix whose columns are rewritten in place (same row pointers, same
addresses, nothing forgotten) is solved with the columns it now has: by the
single solve and the batch, within one workgroup and across several, back and
forth, and where the new columns are too far apart for the one-launch solve.
The results are those of a matrix that was never anything else, bit for bit."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import from_coo

pytestmark = pytest.mark.gpu


def circulant(n, offsets, seed):
    """Rows of 2 len(offsets) + 1 entries whatever the offsets."""
    i = np.arange(n)
    rows = np.concatenate([np.maximum(i, (i + o) % n) for o in offsets])
    cols = np.concatenate([np.minimum(i, (i + o) % n) for o in offsets])
    w = 0.5 + np.random.default_rng(seed).integers(1, 9, len(rows)) / 9.0
    diag = np.bincount(rows, w, n) + np.bincount(cols, w, n) + 0.25
    return from_coo(n, np.concatenate([rows, i]), np.concatenate([cols, i]),
                    np.concatenate([-w, diag]), symmetric=True)


PATTERNS = {
    "one_workgroup": (1000, [1, 2], [3, 400]),
    "own_rows_only": (5003, [1, 2], [1, 3]),
    "far": (5003, [1, 2], [700, 2300]),
    "rows_of_17": (20003, range(1, 9), range(2, 10)),
    "too_far_apart": (20003, range(1, 9), range(1100, 9900, 1100)),
    "near_again": (20003, range(1100, 9900, 1100), range(1, 9)),
}


@pytest.mark.parametrize("name", list(PATTERNS))
def test_single_solve(name):
    n, first, second = PATTERNS[name]
    hosts = [circulant(n, first, 1), circulant(n, second, 2)]
    assert np.array_equal(hosts[0].ia, hosts[1].ia)
    assert not np.array_equal(hosts[0].ja, hosts[1].ja)
    rng = np.random.default_rng(3)
    b, x0 = S.to_dev(rng.standard_normal(n)), S.to_dev(rng.standard_normal(n))
    fresh = [S.DeviceCSR.from_csr(h) for h in hosts]
    precs = [S.make_preconditioner(f, h, "line_jacobi") for f, h in zip(fresh, hosts)]
    want = [S.pcg(f, b, P, tol=1e-10, x0=x0) for f, P in zip(fresh, precs)]
    A = S.DeviceCSR.from_csr(hosts[0])
    for k in (0, 1, 0, 1, 1):
        A.ja.copy_(fresh[k].ja)
        A.a.copy_(fresh[k].a)
        got = S.pcg(A, b, precs[k], tol=1e-10, x0=x0)
        assert got.flag == 0
        if name not in ("too_far_apart", "near_again"):
            assert (got.iterations, got.res0) == (want[k].iterations, want[k].res0), k
            assert torch.equal(got.x, want[k].x), k
        # (a plan that did not fit the earlier columns is not tried again: the
        # launches then add up the dot products in another order.  Either ends
        # with |r| <= 1e-10 |r0|, and the least eigenvalue is 1/4.)
        assert float((got.x - want[k].x).norm()) <= 8.1e-10 * want[k].res0, k


def test_batch():
    sizes = [5003, 1000, 2049, 17, 5003]
    sets = [[circulant(n, o, 7 + k) for k, n in enumerate(sizes)] for o in ([1, 2], [3, 6])]
    rng = np.random.default_rng(4)
    rhs = [rng.standard_normal(n) for n in sizes]
    fresh = [S.Batch.from_systems(s, rhs) for s in sets]
    want = [S.pcg_batched(B, tol=1e-10, block=-1) for B in fresh]
    B = S.Batch.from_systems(sets[0], rhs)
    for k in (0, 1, 0):
        B.A.ja.copy_(fresh[k].A.ja)
        B.A.a.copy_(fresh[k].A.a)
        B.d_r.copy_(fresh[k].d_r)
        got = S.pcg_batched(B, tol=1e-10, block=-1)
        assert torch.equal(got[0], want[k][0]), k
        for i in range(1, 5):
            assert np.array_equal(got[i], want[k][i]), (k, i)
