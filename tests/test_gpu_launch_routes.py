"""The Jacobi solves and lockstep batches that run as one launch, by launches
instead (resident_polls 0): the tests of the launch loop, its graphs, its stops and
its matrix formats, which small systems no longer reach otherwise, and batches of
systems of many row blocks and long rows.  Large solves switch to row classes
with and without graphs, and in batches of one iteration and of five."""
import numpy as np
import pytest

import test_gpu_batched as batched
import test_gpu_pcg as pcg
import test_gpu_vi as vi
from lap_amd import solver as S
from lap_amd.problems import grid_laplacian
from test_gpu_cls import CASES as LARGE, both, same
from test_gpu_rewritten_columns import circulant

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def launches():
    start = S.set_option("resident_polls", 0)
    yield
    S.set_option("resident_polls", start)


test_graphs = pcg.test_pcg_deterministic_and_graph_invariant
test_stops = pcg.test_jacobi_control_flow_edge_cases
test_more_stops = pcg.test_maxit_flag
test_zero = pcg.test_zero_rhs_converges_immediately
test_value_indexed = vi.test_value_indexed_jacobi_pcg_bitwise
test_offset_tables = vi.test_delta_indexed_falls_back
test_offset_limit = vi.test_delta_indexed_offset_limit
test_value_limit = vi.test_value_indexed_table_limit
test_long_rows = vi.test_delta_indexed_edge_rows
test_batch = batched.test_batched_matches_per_system_oracle
test_batch_rows = batched.test_batched_tpr1_rows_are_reference_order


def test_batch_of_many_row_blocks_and_long_rows(orc):
    """Twelve iterations; only the dot products' order differs from the oracle's."""
    systems = [grid_laplacian([130, 101], 0.05), circulant(5003, range(1, 20), 1),
               circulant(3000, range(1, 400), 2), grid_laplacian([1], 0.5),
               grid_laplacian([23, 24, 25], 0.05), circulant(1111, range(1, 9), 3)]
    rng = np.random.default_rng(25)
    rhs = [rng.standard_normal(A.n) for A in systems]
    rhs[5][:] = 0.0
    B = S.Batch.from_systems(systems, rhs)
    x0 = rng.standard_normal(B.A.n)
    x0[-1111:] = 0.0
    x, it, fl, r0, rs, _ = S.pcg_batched(B, tol=1e-30, maxit=11, block=-1, x0=S.to_dev(x0))
    xs = [v.cpu().numpy() for v in B.split(x)]
    for k, (A, b) in enumerate(zip(systems, rhs)):
        if k == 3:  # one row: solved after the first iteration, and 0 / 0 from there on
            off = int(B.row_off[k])
            assert abs(xs[k][0] * A.a[0] - b[0]) <= 2e-15 * (abs(b[0]) + abs(A.a[0] * x0[off]))
            continue
        if k == 5:
            assert it[k] == 0 and fl[k] == 0 and not xs[k].any()
            continue
        off = int(B.row_off[k])
        xo, ito, flo, ho = orc.cg(A, b, "line_jacobi", tol=1e-30, maxit=11,
                                  x0=x0[off:off + A.n].copy())
        assert (it[k], fl[k]) == (ito, flo), k
        assert np.linalg.norm(xs[k] - xo) <= 1e-10 * np.linalg.norm(xo), k
        np.testing.assert_allclose([r0[k], rs[k]], [ho[0], ho[-1]], rtol=1e-10)


@pytest.mark.parametrize("opts", [{"use_graph": 0}, {"graph_iters": 1}, {"graph_iters": 5},
                                  {"use_graph": 0, "graph_iters": 1}])
@pytest.mark.parametrize("solve,kind,mk", [(S.pcg, "line_jacobi", (1, 1)), (S.pcg, "GS_it2", (1, 2)),
                                           (S.pcg, "none", (1, 1)),
                                           (S.pcg_mixed, "line_jacobi", (1, 1)),
                                           (S.pcg_mixed, "none", (1, 1))])
def test_classes_come_in_with_any_batch(opts, solve, kind, mk):
    Ah = LARGE["cube_odd"]()
    b = np.random.default_rng(26).standard_normal(Ah.n)
    kw = {"tol": 1e-9} if solve is S.pcg_mixed else {}
    out = both(Ah, kind, b, maxit=30, mk=mk, solve=solve, **kw, **opts)
    same(*out)
    same(out[0], both(Ah, kind, b, maxit=30, mk=mk, solve=solve, **kw)[0])


def test_not_finite_after_the_classes_came_in():
    """Well conditioned and no tolerance: the residual falls until its square is 0,
    and the next quotient 0 / 0, more than a hundred iterations after the first
    batch of 16."""
    Ah = grid_laplacian([83, 79, 89], 5.0)
    b = np.random.default_rng(27).standard_normal(Ah.n)
    r, s = both(Ah, "line_jacobi", b, maxit=2000)
    assert r.flag == 2 and 100 < r.iterations < 2000
    assert (r.iterations, r.flag) == (s.iterations, s.flag)
    assert np.array_equal(r.history, s.history, equal_nan=True)
    assert np.array_equal(r.x.cpu().numpy(), s.x.cpu().numpy(), equal_nan=True)
