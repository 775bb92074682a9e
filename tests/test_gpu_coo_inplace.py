"""COO -> CSR whose output arrays are the input arrays: ja over rows or cols, a
over vals, whole or shifted, rows of every sort (short, more than 32 and more
than 4096 entries).  The result is the one into arrays of its own, exactly."""
import ctypes as C

import numpy as np
import pytest
import torch

from lap_amd import io as IO
from lap_amd import lib as L
from lap_amd import solver as S

pytestmark = pytest.mark.gpu


def entries(lengths, m, seed):
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(len(lengths)), lengths)
    c = np.concatenate([rng.permutation(m)[:k] for k in lengths])
    o = rng.permutation(len(r))
    return r[o].astype(np.int32), c[o].astype(np.int32), rng.standard_normal(len(r))


@pytest.mark.parametrize("over", ["cols", "rows", "shifted"])
@pytest.mark.parametrize("lengths", [[3] * 40000, [33, 1, 32] * 50, [5000, 4097, 2, 9000]])
def test_outputs_over_the_entries(lengths, over):
    n, m = len(lengths), max(lengths) + 5
    r, c, v = entries(lengths, m, n)
    want = IO.coo_to_csr(n, *(torch.from_numpy(x).to(S.DEV) for x in (r, c, v)), False, m)
    nnz, at = len(r), 7 if over == "shifted" else 0
    ints = {k: torch.zeros(nnz + at, dtype=torch.int32, device=S.DEV) for k in ("rows", "cols")}
    vals = torch.zeros(nnz + at, dtype=torch.float64, device=S.DEV)
    ints["rows"][at:] = torch.from_numpy(r).to(S.DEV)
    ints["cols"][at:] = torch.from_numpy(c).to(S.DEV)
    vals[at:] = torch.from_numpy(v).to(S.DEV)
    ia = torch.empty(n + 1, dtype=torch.int32, device=S.DEV)
    ja = ints["rows" if over == "rows" else "cols"][:nnz]
    torch.cuda.synchronize()
    cnt = C.c_int(0)
    st = L.load().lap_coo_to_csr(n, m, nnz, S.ptr(ints["rows"][at:]), S.ptr(ints["cols"][at:]),
                                 S.ptr(vals[at:]), 0, nnz, S.ptr(ia), S.ptr(ja),
                                 S.ptr(vals[:nnz]), C.byref(cnt))
    assert st == 0 and cnt.value == nnz
    assert torch.equal(ia, want.ia) and torch.equal(ja, want.ja)
    assert torch.equal(vals[:nnz], want.a)


def test_symmetric_diagonal_in_place():
    """The one symmetric matrix whose CSR form has as many entries."""
    n = 70001
    p = torch.randperm(n, generator=torch.Generator().manual_seed(3)).to(torch.int32).to(S.DEV)
    v = torch.arange(n, dtype=torch.float64, device=S.DEV)
    want = v[torch.argsort(p)]
    rows = p.clone()
    ia = torch.empty(n + 1, dtype=torch.int32, device=S.DEV)
    torch.cuda.synchronize()
    cnt = C.c_int(0)
    st = L.load().lap_coo_to_csr(n, n, n, S.ptr(rows), S.ptr(p), S.ptr(v), 1, n, S.ptr(ia),
                                 S.ptr(p), S.ptr(v), C.byref(cnt))
    assert st == 0 and cnt.value == n
    assert torch.equal(p, torch.arange(n, dtype=torch.int32, device=S.DEV))
    assert torch.equal(v, want)
