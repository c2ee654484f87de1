"""y = alpha A x + beta y on node graphs with ragged rows: the streamed product of 2 and 3 equations per node
(row ranges that end inside a workgroup, a row longer than one LDS piece) and the row kernels of 4 (rows
shorter and longer than one trip of loads), beside 1 equation per node.

Bar: every entry within (terms + 3) eps of the dot product of absolute values, eps of the arithmetic."""
import ctypes as C

import numpy as np
import pytest

from coolfluid3_amd import cabi

pytestmark = pytest.mark.gpu


def graph(N, seed):
    """Row 0 couples to every node, the others to 1 to 40 random ones; diagonal included, columns sorted."""
    rng = np.random.default_rng(seed)
    rows = [np.arange(N)] + [np.unique(np.append(rng.integers(0, N, rng.integers(0, 40)), i)) for i in range(1, N)]
    start = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    return start.astype(np.uint32), np.concatenate(rows).astype(np.uint32)


@pytest.mark.parametrize("neq", [1, 2, 3, 4])
@pytest.mark.parametrize("N", [1, 17, 18, 19, 23, 24, 25, 28, 29, 301])
def test_product_on_ragged_rows(neq, N):
    start, cols = graph(N, 10 * N + neq)
    rng = np.random.default_rng(N)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, cols, N))
    s.enable_fp32()
    s.reset(0.3)
    dense = np.zeros((N * neq, N * neq))
    rows = np.repeat(np.arange(N), np.diff(start.astype(np.int64)))
    for r, c in zip(rows, cols):
        dense[r * neq:(r + 1) * neq, c * neq:(c + 1) * neq] = 0.3
    for k in rng.integers(0, len(cols), 150):
        i, j, v = rows[k] * neq + rng.integers(neq), int(cols[k]) * neq + rng.integers(neq), rng.uniform(-2, 2)
        s.set_value(j, i, v)
        dense[i, j] = v
    x, y0 = rng.uniform(-1, 1, N * neq), rng.uniform(-1, 1, N * neq)
    terms = np.diff(start.astype(np.int64)).repeat(neq) * neq
    print("neq", neq, "N", N, flush=True)
    s.set_vector(cabi.SOLUTION, x)
    for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
        s.set_vector(cabi.RHS, y0)
        s.apply_device(alpha, s.vector_ptr(cabi.SOLUTION), beta, s.vector_ptr(cabi.RHS))
        bar = (terms + 3) * 2.0 ** -52 * (abs(alpha) * np.abs(dense) @ np.abs(x) + abs(beta) * np.abs(y0))
        assert (np.abs(s.vector(cabi.RHS) - (alpha * dense @ x + beta * y0)) <= bar).all()
    # FP32: the vectors as floats in the first half of the FP64 buffers
    s.round_fp32()
    x32, y32 = x.astype(np.float32), y0.astype(np.float32)
    pad = np.zeros(2 * N * neq, np.float32)
    pad[:N * neq] = x32
    s.set_vector(cabi.SOLUTION, pad.view(np.float64))
    d32 = dense.astype(np.float32).astype(np.float64)
    for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
        pad[:N * neq] = y32
        s.set_vector(cabi.RHS, pad.view(np.float64))
        s.apply_fp32_device(alpha, s.vector_ptr(cabi.SOLUTION), beta, s.vector_ptr(cabi.RHS))
        got = s.vector(cabi.RHS).view(np.float32)[:N * neq].astype(np.float64)
        bar = (terms + 3) * 2.0 ** -23 * (abs(alpha) * np.abs(d32) @ np.abs(x32) + abs(beta) * np.abs(y32))
        assert (np.abs(got - (alpha * d32 @ x32.astype(np.float64) + beta * y32)) <= bar).all()
    s.close()
    ctx.close()


@pytest.mark.parametrize("neq", [2, 3])
@pytest.mark.parametrize("N", [85, 86, 128, 129, 300])
def test_short_rows_fill_the_workgroups(neq, N):
    """Rows of one or two blocks: a workgroup takes one per thread (85 or 128), the last one what is left."""
    print("neq", neq, "N", N, flush=True)
    two = np.arange(N) % 3 == 1
    start = np.concatenate([[0], np.cumsum(1 + two)]).astype(np.uint32)
    cols = np.concatenate([[i - 1, i] if two[i] else [i] for i in range(N)]).astype(np.uint32)
    rng = np.random.default_rng(N)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, cols, N))
    s.reset(0.25)
    x = rng.integers(-8, 9, N * neq).astype(np.float64)          # the sums are exact
    b = x.reshape(N, neq).sum(1) * 0.25
    y = np.repeat(b + np.where(two, np.roll(b, 1), 0.0), neq)
    s.set_vector(cabi.SOLUTION, x)
    s.apply_device(1.0, s.vector_ptr(cabi.SOLUTION), 0.0, s.vector_ptr(cabi.RHS))
    assert np.array_equal(s.vector(cabi.RHS), y)
    s.close()
    ctx.close()


@pytest.mark.parametrize("neq", [1, 2, 3])
def test_products_are_fused(neq):
    """Row sums are fused multiply-adds in ascending order: with a a = 1 + 2 e + e^2, whose last term the rounded
    product drops, -(1 + 2 e) 1 + a a leaves exactly e^2."""
    print("neq", neq, flush=True)
    N = 30
    other = np.maximum(np.arange(N), 1)                              # row 0: columns 0 and 1; row i: 0 and i
    cols = np.stack([np.zeros(N), other], axis=1).ravel().astype(np.uint32)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(np.arange(N + 1, dtype=np.uint32) * 2, cols, N))
    s.enable_fp32()
    for e, dtype in ((2.0 ** -30, np.float64), (2.0 ** -13, np.float32)):
        s.reset(0.0)
        x = np.ones(N * neq)
        for i in range(N):
            for k in range(neq):
                s.set_value(k, i * neq + k, -(1 + 2 * e))
                s.set_value(int(other[i]) * neq + k, i * neq + k, 1 + e)
                x[other[i] * neq + k] = 1 + e
        if dtype == np.float64:
            s.set_vector(cabi.SOLUTION, x)
            s.apply_device(1.0, s.vector_ptr(cabi.SOLUTION), 0.0, s.vector_ptr(cabi.RHS))
            y = s.vector(cabi.RHS)
        else:
            s.round_fp32()
            pad = np.zeros(2 * N * neq, np.float32)
            pad[:N * neq] = x
            s.set_vector(cabi.SOLUTION, pad.view(np.float64))
            s.apply_fp32_device(1.0, s.vector_ptr(cabi.SOLUTION), 0.0, s.vector_ptr(cabi.RHS))
            y = s.vector(cabi.RHS).view(np.float32)[:N * neq]
        assert (y == e * e).all()
    s.close()
    ctx.close()


def test_product_of_more_rows_than_workgroups():
    """More rows than one launch reaches (2^22 workgroups of 128 rows of one block): the last ones are multiplied
    too."""
    N = 2 ** 29 + 3
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=2, graph=(np.arange(N + 1, dtype=np.uint32), np.arange(N, dtype=np.uint32), N))
    s.reset(0.5)
    s.reset_vector(cabi.SOLUTION, 3.0)
    s.reset_vector(cabi.RHS, 1.0)
    print("system made", flush=True)
    s.apply_device(2.0, s.vector_ptr(cabi.SOLUTION), 1.0, s.vector_ptr(cabi.RHS))
    value = C.c_double()
    for row in (0, N // 2, N - 5, N - 4, N - 3, N - 2, N - 1):
        for eq in (0, 1):
            cabi.check(cabi.lib().cf3hip_vector_get_value(s.h, cabi.RHS, row, eq, C.byref(value)))
            assert value.value == 2.0 * (0.5 * 3.0 + 0.5 * 3.0) + 1.0, (row, eq)
    s.close()
    ctx.close()
