"""Chunked triangular solves at the sizes and values where they can go wrong:
part-filled steps and tiles, one chunk, several workgroups, chains longer than
the results kept in LDS, rows of no, one and four dependencies, and right-hand
sides that leave the refined division's range.  Every result is bitwise the
level launches' (sptrsv_mode 0), through the IC0 preconditioner's application (a
lower and an upper solve)."""
import numpy as np
import pytest
import torch

from lap_amd import solver as S
from lap_amd.problems import from_coo, grid_laplacian

pytestmark = pytest.mark.gpu


def _long_range(n):
    """Entries 1, 700 and 5000 rows back: local, beyond a chunk's recent
    steps, and in another chunk."""
    i = np.arange(n)
    rows, cols = [], []
    for off in (1, 700, 5000):
        rows.append(i[off:])
        cols.append(i[:-off] if off < n else i[:0])
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    keep = (rows * 7 + cols) % 3 != 0  # uneven: rows with 0 to 3 dependencies
    rows, cols = rows[keep], cols[keep]
    w = 0.5 + (rows % 11) / 7.0
    diag = np.bincount(rows, w, n) + np.bincount(cols, w, n) + 0.25
    return from_coo(n, np.concatenate([rows, i]), np.concatenate([cols, i]),
                    np.concatenate([-w, diag]), symmetric=True)


CASES = {
    "one_row": lambda: grid_laplacian([1], 1.0),
    "65_line": lambda: grid_laplacian([65], 0.1),
    "63x2": lambda: grid_laplacian([63, 2], 1e-3),
    "8x8x8": lambda: grid_laplacian([8, 8, 8], 1e-3),
    "9x17x5": lambda: grid_laplacian([9, 17, 5], 1e-3),
    "33x31x40": lambda: grid_laplacian([33, 31, 40], 1e-3),
    "300x7": lambda: grid_laplacian([300, 7], 1e-3),
    "130x131": lambda: grid_laplacian([130, 131], 1e-3),
    "long_range": lambda: _long_range(20011),
}


def _rhs(n, what):
    b = np.random.default_rng(3).standard_normal(n)
    if what == "zeros":  # rows whose sums are exactly zero
        b[: max(1, n // 2)] = 0.0
        b[-1] = -0.0
    elif what == "extremes":  # quotients near and past both ends of the range
        b *= 10.0 ** np.random.default_rng(4).integers(-300, 300, n)
        b[n // 2] = 5e-324
        b[-1] = np.inf
    return S.to_dev(b)


@pytest.mark.parametrize("name", list(CASES))
def test_chunked_solves_equal_the_level_launches(name):
    Ah = CASES[name]()
    A = S.DeviceCSR.from_csr(Ah)
    P = S.make_preconditioner(A, Ah, "ichol")
    prev = S.set_option("sptrsv_mode", 0)
    try:
        for what in ("normal", "zeros", "extremes"):
            print(f"[case] {name} {what}", flush=True)
            r = _rhs(Ah.n, what)
            S.set_option("sptrsv_mode", 0)
            want = S.prec_apply(A, P, r)
            S.set_option("sptrsv_mode", 3)
            for _ in range(2):  # the second solve meets the first one's values in the inboxes
                got = S.prec_apply(A, P, r)
                assert torch.equal(got.view(torch.int64), want.view(torch.int64)) or (
                    torch.equal(got.isnan(), want.isnan()) and
                    torch.equal(got.nan_to_num(0.0).view(torch.int64),
                                want.nan_to_num(0.0).view(torch.int64)))
    finally:
        S.set_option("sptrsv_mode", prev)
