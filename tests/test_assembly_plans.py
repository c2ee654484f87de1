"""The block-list assembly of the specialised triangles and tetrahedra at the limits of its plans, against the
oracle: fans whose centre rows fill a workgroup's 128 block lists exactly, miss them by one (the staged
reduction then serves the system), or fit easily; single elements; periodic links, where a block sums several
mesh nodes that hold different states.

Bars: FP64 row-relative 1e-12 as everywhere; FP32 1e-6 of the element matrices plus one rounding per summed
contribution."""
import time

import numpy as np
import pytest

from coolfluid3_amd import cabi, cases, meshgen
from oracle import pyoracle
from tests.test_gpu_parity import gpu_case, oracle_system, row_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cabi.Context(0)
    yield c
    c.close()


def case_of(etype, coords, conn, periodic=None, seed=5):
    rng = np.random.default_rng(seed)
    N, dim = coords.shape
    return cases.Case("fan", etype, coords, conn.astype(np.uint32), None, 1e-2, 1e-2, u0=rng.uniform(-1, 1, (N, dim)),
                      p0=rng.uniform(-1, 1, N), periodic=periodic)


def triangle_fan(n):
    """n triangles around node 0, its local index rotating."""
    a = 2 * np.pi * np.arange(n) / n
    coords = np.concatenate([[[0.3, 0.2]], np.stack([0.3 + np.cos(a), 0.2 + np.sin(a)], axis=1)])
    conn = np.stack([np.zeros(n, int), 1 + np.arange(n), 1 + (np.arange(n) + 1) % n], axis=1)
    return case_of(cabi.TRIAG2D, coords, np.stack([np.roll(c, i % 3) for i, c in enumerate(conn)]))


def tetrahedron_fan(n):
    """n tetrahedra around the edge of nodes 0 and 1, their local indices changing by even permutations."""
    a = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(a), np.sin(a), np.zeros(n)], axis=1)
    coords = np.concatenate([[[0, 0, -0.5], [0, 0, 0.5]], ring]) + 0.1
    conn = np.stack([np.zeros(n, int), 2 + np.arange(n), 2 + (np.arange(n) + 1) % n, np.ones(n, int)], axis=1)
    even = np.array([[0, 1, 2, 3], [1, 0, 3, 2], [2, 3, 0, 1], [3, 2, 1, 0]])
    return case_of(cabi.TETRA3D, coords, np.stack([c[even[i % 4]] for i, c in enumerate(conn)]))


# triangles: 32 + 96 = 128 lists, 33 + 97 = 130; tetrahedra: 96 + 16 + 16 = 128, 97 + 17 + 17 = 131
@pytest.mark.parametrize("make,n", [(triangle_fan, 3), (triangle_fan, 95), (triangle_fan, 96), (triangle_fan, 97),
                                    (tetrahedron_fan, 3), (tetrahedron_fan, 95), (tetrahedron_fan, 96),
                                    (tetrahedron_fan, 97)])
def test_fans_at_the_list_limit(ctx, oracle, make, n):
    print(make.__name__, n, flush=True)
    case = make(n)
    neq = case.dim + 1
    start, _, _, vref, rref = oracle_system(oracle, case, theta=0.7)
    g = gpu_case(ctx, case, theta=0.7, fp32=True)
    g.assemble(cabi.FP64)
    v, r = g.system.values(), g.system.vector(cabi.RHS)
    assert row_rel_err(v, vref, neq, start) <= 1e-12
    assert np.abs(r - rref).max() <= 1e-12 * np.abs(rref).max()
    g.assemble(cabi.FP64)
    assert np.array_equal(g.system.values(), v) and np.array_equal(g.system.vector(cabi.RHS), r)
    g.assemble(cabi.FP32)
    assert row_rel_err(g.system.values_fp32().astype(np.float64), vref, neq, start) <= 1e-6 + n * 2.0 ** -24
    g.close()


@pytest.mark.parametrize("etype,n", [(cabi.TRIAG2D, 2), (cabi.TRIAG2D, 5), (cabi.TETRA3D, 2), (cabi.TETRA3D, 4)])
def test_periodic_blocks_of_several_nodes(ctx, oracle, etype, n):
    """Periodic in every direction, with states that differ between the linked nodes; at n = 2 an element
    can hold two nodes of one block row."""
    print(etype, n, flush=True)
    dim = 2 if etype == cabi.TRIAG2D else 3
    coords, conn = meshgen.rect_tris(n, n) if dim == 2 else meshgen.box_tetras(n, n, n)
    faces = [(np.flatnonzero(coords[:, d] > 1 - 1e-12), np.flatnonzero(coords[:, d] < 1e-12), -np.eye(dim)[d])
             for d in range(dim)]
    case = case_of(etype, coords, conn, periodic=cases.periodic_links(coords, faces))
    p2m = cases.periodic_p2m(*case.periodic)
    start, cols, slots = oracle.build_sparsity(p2m[case.conn], int(p2m.max()) + 1)
    et = pyoracle.TRIAG2D if dim == 2 else pyoracle.TETRA3D
    ua = oracle.linearize_u(case.u0, case.u0, case.u0, case.u0)
    vref, rref = oracle.ns_assemble_p2m(et, pyoracle.ns_params(dt=case.dt, theta=0.7), coords, case.conn, p2m, case.u0,
                                        case.p0, ua, np.full(case.n_nodes, case.nu), start, slots)
    g = gpu_case(ctx, case, theta=0.7)
    g.assemble(cabi.FP64)
    assert np.abs(g.system.values() - vref).max() <= 1e-12 * np.abs(vref).max()
    assert np.abs(g.system.vector(cabi.RHS) - rref).max() <= 1e-12 * np.abs(rref).max()
    g.close()


@pytest.mark.parametrize("etype", [cabi.TRIAG2D, cabi.TETRA3D])
def test_infinite_tau_argument(ctx, oracle, etype):
    """Velocities whose squares overflow: tau = 1 / sqrt(inf) = 0, so a continuity row is the divergence sum over
    elements of V / (dim + 1) grad N_b alone, and finite (the momentum rows hold tau_bulk = inf)."""
    print(etype, flush=True)
    coords, conn = meshgen.rect_tris(3, 3) if etype == cabi.TRIAG2D else meshgen.box_tetras(2, 2, 2)
    case = case_of(etype, coords, conn)
    case.u0 *= 1e160
    d, k, X = case.dim, case.dim + 1, case.coords[case.conn]
    start, _, slots = oracle.build_sparsity(case.conn, case.n_nodes)
    grad = np.linalg.inv(X[:, 1:] - X[:, :1]).transpose(0, 2, 1)
    grad = np.concatenate([-grad.sum(1, keepdims=True), grad], axis=1)
    vol = np.abs(np.linalg.det(X[:, 1:] - X[:, :1])) / (2 if d == 2 else 6)
    div = (vol / k)[:, None, None] * grad
    ref = np.zeros((int(start[-1]), k))
    np.add.at(ref[:, :d], slots.reshape(-1, k, k), np.broadcast_to(div[:, None], (len(div), k, k, d)))
    rref = np.zeros(case.n_nodes)
    np.add.at(rref, case.conn, -np.einsum("ebi,ebi->e", div, case.u0[case.conn])[:, None])
    g = gpu_case(ctx, case, theta=0.7)
    g.assemble(cabi.FP64)
    v, r = g.system.values().reshape(-1, k, k)[:, d], g.system.vector(cabi.RHS).reshape(-1, k)[:, d]
    assert np.abs(v - ref).max() <= 1e-12 * np.abs(ref).max()
    assert np.abs(r - rref).max() <= 1e-12 * np.abs(rref).max()
    g.close()


@pytest.mark.parametrize("n", [129, 5000, 70000])
def test_periodic_hub_is_refused(ctx, n):
    """All nodes of a ring linked to one: a block row of 2 n incidences and n column nodes, far above what a
    workgroup holds (and, at n = 5000 and 70000, above the 12 bits of an incidence number in the contribution
    lists), is refused at once."""
    print(n, flush=True)
    case = triangle_fan(n)
    links = np.ones(n + 1, np.uint32)
    active = (np.arange(n + 1) > 1).astype(np.uint8)
    mesh = cabi.Mesh(ctx, case.etype, case.coords, case.conn)
    t = time.perf_counter()
    with pytest.raises(cabi.Cf3HipError, match="incident elements"):
        cabi.System(ctx, mesh, periodic=(links, active))
    assert time.perf_counter() - t < 2
    mesh.close()


def test_plans_only_where_they_are_read(ctx):
    """The specialised kernels take dim + 1 equations: systems of other sizes hold no plans (about 100 bytes a node
    of a triangle mesh, 350 of tetrahedra)."""
    for coords, conn, etype, least in ((*meshgen.rect_tris(24, 24), cabi.TRIAG2D, 60),
                                       (*meshgen.box_tetras(8, 8, 8), cabi.TETRA3D, 200)):
        mesh = cabi.Mesh(ctx, etype, coords, conn)
        N, full = len(coords), coords.shape[1] + 1
        extra = {}
        for neq in (1, 2, full):
            before = ctx.memory()
            s = cabi.System(ctx, mesh, neq=neq)
            extra[neq] = ctx.memory() - before - 8 * (s.n_blocks * neq * neq + 2 * N * neq)
            s.close()
        print(N, extra, flush=True)
        assert extra[1] == extra[2] and extra[full] >= extra[1] + least * N
        mesh.close()


def test_batch_with_systems_beyond_the_plans(ctx):
    """Systems with a row that no plan holds, in a batch with others (first, between, last, alone): every system
    gets the bits of its own single assembly."""
    def make(case):
        g = gpu_case(ctx, case, fp32=True)
        g.assemble(cabi.FP32)
        return g, g.system.values_fp32()
    hub = [make(tetrahedron_fan(97)) for _ in range(3)]
    tets = [make(case_of(cabi.TETRA3D, *meshgen.box_tetras(n, n, n), seed=n)) for n in (3, 6)]
    batch = cabi.Batch(ctx, 5)
    for group in ([hub[0]] + tets, [tets[0], hub[0], tets[1]], tets + [hub[0]], [hub[0]], hub, [tets[1]],
                  [hub[0], tets[0], hub[1], tets[1], hub[2]]):
        print(len(group), flush=True)
        for g, _ in group:
            g.system.reset(7.0)
            g.system.round_fp32()
        prms = [cabi.NSParams.from_buffer_copy(g.prm) for g, _ in group]
        for p in prms:
            p.precision = cabi.FP32
        batch.assemble([g.system for g, _ in group], [g.fields for g, _ in group], prms)
        for g, ref in group:
            assert np.array_equal(g.system.values_fp32(), ref)
    batch.close()
    for g, _ in hub + tets:
        g.close()
