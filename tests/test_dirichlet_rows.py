"""Symmetric Dirichlet conditions on ragged rows (shorter and longer than the 16 blocks a lane group takes at
once) against the oracle: several calls between resets, dofs repeated within and across calls, every dof of a
node or one of them, and a reset in between.

Bar: values exactly (entries are kept, zeroed or set to 1); rhs within (blocks of a row x neq + 2) eps of the
sum of the absolute terms, whose order is the kernel's own."""
import ctypes as C

import numpy as np
import pytest

from coolfluid3_amd import cabi

pytestmark = pytest.mark.gpu


def symmetric_graph(N, seed):
    rng = np.random.default_rng(seed)
    a = np.eye(N, dtype=bool)
    a[0, :] = a[:, 0] = True                       # a hub: one row as long as the system
    for i, j in rng.integers(0, N, (3 * N, 2)):
        a[i, j] = a[j, i] = True
    rows = [np.flatnonzero(r) for r in a]
    start = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    return start.astype(np.uint32), np.concatenate(rows).astype(np.uint32)


@pytest.mark.parametrize("neq", [1, 2, 3, 4])
@pytest.mark.parametrize("N", [1, 17, 200])
def test_conditions_against_oracle(oracle, neq, N):
    print("neq", neq, "N", N, flush=True)
    start, cols = symmetric_graph(N, N + neq)
    rng = np.random.default_rng(N)
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=neq, graph=(start, cols, N))
    n = int(start[-1])
    for _ in range(2):                              # the second round after a reset
        s.reset(0.0)
        for i in range(N):                          # distinct values, one block row at a time
            idx = cols[start[i]:start[i + 1]]
            for c in idx:
                s.set_value(int(c) * neq + int(rng.integers(neq)), i * neq + int(rng.integers(neq)), rng.uniform(-2, 2))
        vals = s.values()
        rhs, sol = rng.uniform(-1, 1, N * neq), rng.uniform(-1, 1, N * neq)
        s.set_vector(cabi.RHS, rhs)
        s.set_vector(cabi.SOLUTION, sol)
        scale = np.abs(rhs) + 3 * np.abs(vals).max() * np.diff(start.astype(np.int64)).max() * neq
        for call in range(3):
            k = max(1, N // 4)
            nodes = rng.integers(0, N, k).astype(np.uint32)
            nodes = np.concatenate([nodes, nodes[:2], np.zeros(1 if call == 1 else 0, np.uint32)]).astype(np.uint32)
            eqs = rng.integers(0, neq, len(nodes)).astype(np.uint32)
            v = rng.uniform(-1, 1, len(nodes))
            s.dirichlet(nodes, eqs, v)
            oracle.dirichlet(neq, start, cols, vals, rhs, sol, nodes, eqs, v)
            assert np.array_equal(s.values(), vals)
            assert np.array_equal(s.vector(cabi.SOLUTION), sol)
            bar = (np.diff(start.astype(np.int64)).max() * neq + 2) * 2.0 ** -52 * scale
            assert (np.abs(s.vector(cabi.RHS) - rhs) <= bar).all()
    assert n == s.n_blocks
    s.close()
    ctx.close()


def test_more_rows_than_lanes_in_32_bits():
    """A condition that a row past 2^28 couples to (16 lanes per row: more than 2^32 lanes): identities but for the
    last row, which holds the column of the one before it."""
    N = 2 ** 28 + 5
    start = np.arange(N + 1, dtype=np.uint32)
    start[N] += 1
    cols = np.arange(N + 1, dtype=np.uint32)
    cols[N - 1], cols[N] = N - 2, N - 1
    ctx = cabi.Context(0)
    s = cabi.System(ctx, neq=1, graph=(start, cols, N))
    del start, cols
    s.reset(2.0)
    s.reset_vector(cabi.RHS, 1.0)
    print("system made", flush=True)
    s.dirichlet([N - 2], [0], [3.0])
    value = C.c_double()

    def rhs(row):
        cabi.check(cabi.lib().cf3hip_vector_get_value(s.h, cabi.RHS, row, 0, C.byref(value)))
        return value.value
    assert s.get_value(N - 2, N - 1) == 0.0 and rhs(N - 1) == 1.0 - 2.0 * 3.0
    assert s.get_value(N - 2, N - 2) == 1.0 and rhs(N - 2) == 3.0
    assert s.get_value(0, 0) == 2.0 and rhs(0) == 1.0
    s.close()
    ctx.close()
