"""The three-launch BiCGStab iteration of small systems, 1 to 4 equations per node: rows of 1 to 13 blocks, graphs
whose rows are no multiple of a workgroup's, odd and even iteration counts at the stops, in FP64 and in the
precision form on stored FP32 values (residual replacements at any parity); and couplings in all rows on either
side of the limits in block rows.

Bars: converged, and the true residual on the matrix read back meets the tolerance to within the drift of the
recursive residual (a factor 10, as in the other solver tests)."""
import ctypes as C

import numpy as np
import pytest

from coolfluid3_amd import cabi

pytestmark = pytest.mark.gpu


# one row, a few rows, rows just above a workgroup's 16 or 32, and thousands (20000: the five-launch form)
@pytest.mark.parametrize("neq,N", [(q, n) for q in (1, 2, 3, 4) for n in (1, 3, 33, 700, 6000)] + [(2, 20000)])
def test_solves_across_sizes(neq, N):
    print("neq", neq, "N", N, flush=True)
    rng = np.random.default_rng(N + neq)
    rows = [np.unique(np.append(rng.integers(0, N, min(N, int(rng.integers(0, 13)))), i)) for i in range(N)]
    start = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    cols = np.concatenate(rows).astype(np.uint32)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, cols, N))
    s.enable_fp32()
    s.reset(-0.02)                                   # weak couplings, then a dominant diagonal that varies
    for i in range(min(N, 700)):
        for e in range(neq):
            s.set_value(i * neq + e, i * neq + e, 1.0 + 3.0 * rng.random())
    for i in range(700, N):
        s.set_row(i, int(rng.integers(neq)), 1.5, 0.0)
    if N > 700:                                      # rows beyond: identity rows in every equation
        for i in range(700, N):
            for e in range(neq):
                s.set_row(i, e, 2.0, 0.0)
    b = rng.uniform(-1, 1, N * neq)
    s.set_vector(cabi.RHS, b)
    rp, ci, v = s.debug_data()
    r64 = np.repeat(np.arange(N * neq), np.diff(rp.astype(np.int64)))

    def residual(x):
        return np.linalg.norm(b - np.bincount(r64, v * x[ci], N * neq)) / np.linalg.norm(b)
    for tol in (1e-3, 1e-7, 1e-12):                  # stops after different, odd and even, counts
        s.reset_vector(cabi.SOLUTION)
        st = s.solve(cabi.solver_params(tol=tol, max_iter=500))
        assert st.converged and residual(s.vector(cabi.SOLUTION)) <= 10 * tol, (tol, st.iterations)
        x = s.vector(cabi.SOLUTION)
        s.reset_vector(cabi.SOLUTION)
        assert s.solve(cabi.solver_params(tol=tol, max_iter=500)).iterations == st.iterations
        assert np.array_equal(s.vector(cabi.SOLUTION), x)
    s.round_fp32()
    for tol in (1e-5, 1e-11):
        s.reset_vector(cabi.SOLUTION)
        st = s.solve(cabi.solver_params(tol=tol, max_iter=500, precision=cabi.FP32))
        assert st.converged and residual(s.vector(cabi.SOLUTION)) <= 10 * tol
    s.close()
    ctx.close()


# block rows up to which an iteration takes three launches
@pytest.mark.parametrize("neq,limit", [(1, 45000), (2, 16000), (3, 9000), (4, 11000)])
@pytest.mark.parametrize("above", [0, 1])
def test_either_side_of_the_limits(neq, limit, above):
    """Rows of 3 to 5 blocks with couplings everywhere and a diagonal that varies, at the limit and one row above."""
    N = limit + above
    print("neq", neq, "N", N, flush=True)
    rng = np.random.default_rng(neq)
    far = 137
    rows = [[j for j in (i - far, i - 1, i, i + 1, i + far) if 0 <= j < N] for i in range(N)]
    start = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, np.concatenate(rows).astype(np.uint32), N))
    s.enable_fp32()
    s.reset(-0.12 / neq)
    diag = rng.uniform(0.7, 2.0, N * neq)
    cabi.check(cabi.lib().cf3hip_matrix_set_diagonal(s.h, diag.ctypes.data_as(C.c_void_p)))
    b = rng.uniform(-1, 1, N * neq)
    s.set_vector(cabi.RHS, b)
    s.round_fp32()
    rp, ci, v = s.debug_data()
    r64 = np.repeat(np.arange(N * neq), np.diff(rp.astype(np.int64)))
    assert np.array_equal(v[(r64 == ci)], diag)
    for prec in (cabi.FP64, cabi.FP32):
        for tol in (1e-4, 1e-11):
            s.reset_vector(cabi.SOLUTION)
            st = s.solve(cabi.solver_params(tol=tol, max_iter=500, precision=prec))
            x = s.vector(cabi.SOLUTION)
            res = np.linalg.norm(b - np.bincount(r64, v * x[ci], N * neq)) / np.linalg.norm(b)
            assert st.converged and st.iterations > 2 and res <= 10 * tol, (prec, tol, st.iterations, res)
    s.close()
    ctx.close()


@pytest.mark.parametrize("neq", [1, 2, 3])
def test_products_are_fused(neq):
    """The row sums of the three-launch iteration are fused multiply-adds: row 0 is the identity and two couplings of
    one lane (8 or 16 blocks apart) whose products with the first direction, -(1 + 2 e) and (1 + e)^2, leave e^2
    (rounded products leave nothing).  All other rows are identities, so alpha = omega = 1 and the first iteration
    ends with x_0 = -e^2."""
    print("neq", neq, flush=True)
    N, far, e = 40, 1 + (8 if neq == 1 else 16), 2.0 ** -30
    rows = [np.arange(N)] + [np.array([0, i]) for i in range(1, N)]
    start = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, np.concatenate(rows).astype(np.uint32), N))
    s.reset(0.0)
    for i in range(N * neq):
        s.set_value(i, i, 1.0)
    s.set_value(neq, 0, -(1 + 2 * e))
    s.set_value(far * neq, 0, 1 + e)
    b = np.zeros(N * neq)
    b[neq], b[far * neq] = 1.0, 1 + e
    s.set_vector(cabi.RHS, b)
    s.reset_vector(cabi.SOLUTION)
    s.solve(cabi.solver_params(tol=1e-60, max_iter=1), raise_on_failure=False)
    x = s.vector(cabi.SOLUTION)
    b[0] = -e * e
    assert np.array_equal(x, b)
    s.close()
    ctx.close()
