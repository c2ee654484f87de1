"""The three-launch BiCGStab iteration of small systems on either side of its size limits, 1 to 4 equations per
node: rows of 1 to 40 blocks, a graph whose rows are no multiple of a workgroup's, odd and even iteration counts at
the stops, in FP64 and in the precision form on stored FP32 values (residual replacements at any parity).

Bars: converged, and the true residual on the matrix read back meets the tolerance to within the drift of the
recursive residual (a factor 10, as in the other solver tests)."""
import numpy as np
import pytest

from coolfluid3_amd import cabi

pytestmark = pytest.mark.gpu


# one row, a few rows, rows just above a workgroup's 16 or 32, and about 40 k / 130 k blocks (beyond the limit of
# 3 and 2 equations per node, below that of 1 and 4)
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
