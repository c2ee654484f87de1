"""The work that a program using cf3hip has it do: assemblies with a product of the assembled operator,
implicit time steps, semi-implicit steps and the serving loop, each through the public Python layer
(coolfluid3_amd.cabi, .cases, .serving) over the range of sizes of the benchmark configurations.

Kinds of case:
  assemble  LinearizeU + Assembly (ZeroLSS, element matrices, scatter, rhs) + one product A x, the loop of
            a program that brings its own Krylov method; asynchronous, inputs resident, as bench.py times it
  step      one implicit step from given fields on a mesh that stays: LinearizeU, Assembly, conditions,
            Krylov solve, update; fields come from and go to host arrays, as cases.GpuCase does it.  Solved
            to 1e-11, a digit below the workloads' default: two solves of one system, each stopped anywhere
            below the tolerance, then give fields that agree to about 1e-6 and better
  si        one semi-implicit step (two inner passes) from given fields
  serve     a few requests through serving.Server: meshes, sparsity, batched assemblies and solves
"""
import math

import numpy as np
import torch

from coolfluid3_amd import cabi, cases, meshgen, serving

ETYPE = {"tri": cabi.TRIAG2D, "tet": cabi.TETRA3D, "hex": cabi.HEXA3D, "quad": cabi.QUAD2D, "prism": cabi.PRISM3D}
NODES = {"tri": 3, "tet": 4, "hex": 8, "quad": 4, "prism": 6}
DEV = "cuda"


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # the 32 x 32 triangle cavity of the reference's acceptance runs: latency and launches
        dict(name="tri_assemble_32", kind="assemble", cell="tri", n=32, spec=True, fp32=False, skew=False),
        # the size of an ordinary serving request, in the precision form (FP32 element matrices)
        dict(name="tet_fp32_assemble_23", kind="assemble", cell="tet", n=23, spec=True, fp32=True, skew=False),
        # the FP64 drop-in's size (64^3 cells), odd: ragged workgroups everywhere
        dict(name="tet_assemble_61", kind="assemble", cell="tet", n=61, spec=True, fp32=False, skew=False),
        # the headline mesh: 128^3 x 6 tetrahedra, 1 % flattened
        dict(name="tet_assemble_128", kind="assemble", cell="tet", n=128, spec=True, fp32=False, skew=True),
        # a large precision-form system
        dict(name="tet_fp32_assemble_100", kind="assemble", cell="tet", n=100, spec=True, fp32=True, skew=True),
        # Q1 hexahedra: the cavity mesh of the Picard configuration, at half its side
        dict(name="hex_assemble_80", kind="assemble", cell="hex", n=80, spec=False, fp32=False, skew=False),
        # 512^2 quadrilaterals, the scaled Taylor-Green mesh, generic expression
        dict(name="quad_assemble_512", kind="assemble", cell="quad", n=512, spec=False, fp32=False, skew=False),
        # the cavity step: GMRES(30) + ILU(0)
        dict(name="cavity_step_32", kind="step", flow="cavity", n=32, fp32=False),
        # the drop-in step: FP64, BiCGStab + Jacobi
        dict(name="cube_step_64", kind="step", flow="cube", n=64, fp32=False),
        # a mid-sized channel step in the precision form
        dict(name="channel_fp32_step_37", kind="step", flow="channel", n=37, fp32=True),
        # semi-implicit Taylor-Green step: BiCGStab on systems of two and of one equation per node
        dict(name="si_step_128", kind="si", n=128),
        # a stretch of the serving loop: eight requests of 12 to 28 cells per side, three steps each
        dict(name="serve_8", kind="serve", count=8, lo=12, hi=28, steps=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["assemble"] * 6 + ["step"] * 4 + ["si", "serve"])
    if kind == "assemble":
        cell = rng.choice(["tri", "tet", "tet", "tet", "hex", "hex", "quad", "prism"])
        lo, hi = {"tri": (16, 700), "tet": (10, 110), "hex": (8, 80), "quad": (16, 700), "prism": (8, 64)}[cell]
        simplex = cell in ("tri", "tet")
        return dict(kind=kind, cell=cell, n=_log(rng, lo, hi), spec=simplex and rng.random() < 0.8,
                    fp32=rng.random() < 0.4, skew=cell == "tet" and rng.random() < 0.3)
    if kind == "step":
        flow = rng.choice(["cavity", "cube", "channel", "channel"])
        if flow == "cavity":
            return dict(kind=kind, flow=flow, n=_log(rng, 12, 36), fp32=False)
        return dict(kind=kind, flow=flow, n=_log(rng, 12, 60), fp32=flow == "channel" and rng.random() < 0.7)
    if kind == "si":
        return dict(kind=kind, n=2 * _log(rng, 16, 100))
    lo = _log(rng, 10, 16)
    return dict(kind=kind, count=rng.randint(3, 8), lo=lo, hi=lo + rng.randint(2, 12), steps=rng.randint(2, 3))


# ------------------------------------------------------------------------------------------------
# what a program has in hand
# ------------------------------------------------------------------------------------------------
class Handles:
    """The framework's handles of one state, closed (in reverse order) when nothing refers to them any more."""

    def __init__(self):
        self.open = []

    def __del__(self):
        while self.open:
            self.open.pop().close()


class State:
    def __init__(self, kind):
        self.kind = kind
        self.handles = Handles()

    def own(self, h):
        self.handles.open.append(h)
        return h


class _Device:
    """A device vector of the framework as torch sees it; a tensor made from it keeps the handles open."""

    def __init__(self, handles, ptr, n):
        self.handles = handles
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": "<f8", "version": 2}


def _flow(case, seed):
    """The cases.Case of an assemble or step case."""
    n = case["n"]
    if case["kind"] == "step":
        if case["flow"] == "cavity":
            f = cases.lid_cavity_2d(n, seed=seed)
        elif case["flow"] == "cube":
            f = cases.inflow_cube_tets(n, seed=seed)
        else:
            f = cases.inflow_cube_tets(n, seed=seed, nu=5e-3, dt=1e-2, amp=0.05, outlet=True)
        f.tol = 1e-11
        return f
    cell = case["cell"]
    if cell == "tri":
        return cases.lid_cavity_2d(n, seed=seed)
    if cell == "tet":
        return cases.inflow_cube_tets(n, seed=seed, nu=5e-4, skew=case["skew"], outlet=True)
    if cell == "hex":
        return cases.lid_cavity_cube_hexas(n, seed=seed, random_velocity=True)
    if cell == "prism":
        return cases.lid_cavity_cube_prisms(n, seed=seed, random_velocity=True)
    coords, conn = meshgen.rect_quads(n, n)
    coords, used = meshgen.jitter(coords, (n, n), 0.1, seed)
    N = coords.shape[0]
    u0 = meshgen.uniform(seed, 2 * N, -1.0, 1.0, offset=used).reshape(N, 2)
    return cases.Case("quads_%d" % n, cabi.QUAD2D, coords, conn, (n, n), 1e-3, 4e-3, theta=0.5, u0=u0, p0=np.zeros(N))


def _pressure(flow, seed):
    return meshgen.uniform(seed + 1, flow.n_nodes, -1.0, 1.0)


def _vector(flow, seed, fp32):
    x = meshgen.uniform(seed + 2, flow.n_nodes * (flow.dim + 1), -1.0, 1.0)
    return x.astype(np.float32) if fp32 else x


def _start_time(seed):
    return float(meshgen.uniform(seed, 1, 0.0, 1.0)[0])


def prepare(case, seed):
    s = State(case["kind"])
    s.case = case
    if case["kind"] == "serve":
        k = case["count"]
        r = meshgen.uniform(seed, 2 * k, 0.0, 1.0).reshape(k, 2)
        cells = [int(round(case["lo"] * (case["hi"] / case["lo"]) ** (i / max(k - 1, 1)))) for i in range(k)]
        s.requests = [serving.Request(i, 0.0, c, 10.0 + 990.0 * r[i, 0], 0.1 * r[i, 1], steps=case["steps"])
                      for i, c in enumerate(cells)]
        s.server = serving.Server(seed=seed, keep_fields=True)
        return s
    s.ctx = s.own(cabi.Context(0))
    if case["kind"] == "si":
        s.flow = f = cases.taylor_green_case(case["n"])
        s.t0 = _start_time(seed)
        s.u0, s.p0 = cases.taylor_green_exact(f.coords, s.t0)
        s.mesh = s.own(cabi.Mesh(s.ctx, f.etype, f.coords, f.conn))
        us = s.own(cabi.System(s.ctx, s.mesh, neq=2, periodic=f.periodic))
        ps = s.own(cabi.System(s.ctx, s.mesh, neq=1, periodic=f.periodic))
        s.fields = s.own(cabi.Fields(s.mesh))
        s.si = s.own(cabi.SemiImplicit(us, ps))
        s.prm = cabi.ns_params(dt=f.dt, theta=f.theta)
        s.solver = cabi.solver_params(cabi.BICGSTAB_JACOBI, tol=1e-13, max_iter=20000)
        s.center = f.bc_regions[0][1]
        s.pvalue = cases.taylor_green_exact(f.coords[s.center], s.t0 + f.dt)[1]
        return s
    s.flow = f = _flow(case, seed)
    prec = cabi.FP32 if case["fp32"] else cabi.FP64
    if case["kind"] == "step":
        s.gpu = s.own(cases.GpuCase(s.ctx, f, precision=prec))
        return s
    f.p0 = _pressure(f, seed)
    s.gpu = s.own(cases.GpuCase(s.ctx, f, precision=prec, use_specializations=case["spec"]))
    s.prm = cabi.ns_params(rho=f.rho, dt=f.dt, theta=f.theta, use_specializations=case["spec"], precision=prec)
    s.x = torch.from_numpy(_vector(f, seed, case["fp32"])).to(DEV)
    s.y = torch.zeros_like(s.x)
    dofs = s.gpu.system.dofs
    s.rhs = torch.as_tensor(_Device(s.handles, s.gpu.system.vector_ptr(cabi.RHS), dofs), device=DEV)
    torch.cuda.synchronize()
    s.ctx.set_async(True)
    return s


def run(s):
    if s.kind == "assemble":
        system = s.gpu.system
        s.gpu.fields.linearize()
        system.assemble(s.gpu.fields, s.prm)
        if s.case["fp32"]:
            system.apply_fp32_device(1.0, s.x.data_ptr(), 0.0, s.y.data_ptr())
            return {"y": s.y}
        system.apply_device(1.0, s.x.data_ptr(), 0.0, s.y.data_ptr())
        return {"y": s.y, "rhs": s.rhs}
    if s.kind == "step":
        g, f = s.gpu, s.flow
        g.fields.set(cabi.FIELD_U, f.u0)
        g.fields.set(cabi.FIELD_P, f.p0)
        g.fields.initialize(f.nu)
        g.u, g.p = f.u0, f.p0
        g.system.reset_vector(cabi.SOLUTION)
        g.step()
        return {"u": g.u, "p": g.p}
    if s.kind == "si":
        s.fields.set(cabi.FIELD_U, s.u0)
        s.fields.set(cabi.FIELD_P, s.p0)
        s.fields.initialize(s.flow.nu)
        s.si.initial(s.fields, s.prm)
        s.si.step(s.fields, s.prm, s.solver, s.solver, pbc=(s.center, s.pvalue))
        return {"u": s.fields.get(cabi.FIELD_U), "p": s.fields.get(cabi.FIELD_P)}
    records, _ = s.server.run(s.requests)
    return {"u%d" % r.rid: r.u for r in records} | {"p%d" % r.rid: r.p for r in records}


# ------------------------------------------------------------------------------------------------
# bytes and operations that a pass cannot do without
# ------------------------------------------------------------------------------------------------
def _sizes(cell, n):
    """nodes, elements and node blocks of the structured meshes."""
    if cell == "tri":
        return (n + 1) ** 2, 2 * n * n, (n + 1) ** 2 + 2 * (3 * n * n + 2 * n)
    if cell == "quad":
        return (n + 1) ** 2, n * n, (3 * n + 1) ** 2
    if cell == "tet":
        return (n + 1) ** 3, 6 * n ** 3, (n + 1) ** 3 + 2 * (7 * n ** 3 + 9 * n * n + 3 * n)
    if cell == "hex":
        return (n + 1) ** 3, n ** 3, (3 * n + 1) ** 3
    return (n + 1) ** 3, 2 * n ** 3, ((n + 1) ** 2 + 2 * (3 * n * n + 2 * n)) * (3 * n + 1)


def _assembly_work(cell, n, vb):
    N, E, nb = _sizes(cell, n)
    k = NODES[cell]
    dim = 2 if cell in ("tri", "quad") else 3
    neq = dim + 1
    # node records in, connectivity in, values and rhs out; one pass of element integrals
    b = N * (3 * dim * 8 + 16) + E * k * 4 + nb * neq * neq * vb + N * neq * 8
    points = 1 if k == dim + 1 else {"quad": 4, "prism": 6, "hex": 8}[cell]
    f = E * (300 + k * k * (neq * neq * 2 + points * 40))
    return b, f


def _product_work(cell, n, vb):
    N, _, nb = _sizes(cell, n)
    neq = 3 if cell in ("tri", "quad") else 4
    return nb * (neq * neq * vb + 4) + N * (4 + 2 * neq * vb), 2 * nb * neq * neq


def _step_work(n, cell, vb, iterations, products):
    b, f = _assembly_work(cell, n, vb)
    pb, pf = _product_work(cell, n, vb)
    return b + iterations * products * pb, f + iterations * products * pf


def work(case):
    if case["kind"] == "assemble":
        vb = 4 if case["fp32"] else 8
        b, f = _assembly_work(case["cell"], case["n"], vb)
        pb, pf = _product_work(case["cell"], case["n"], vb)
        return {"bytes": b + pb, "flops": f + pf}
    if case["kind"] == "step":
        # iterations: about those the present method takes; each reads the matrix once per product
        n = case["n"]
        if case["flow"] == "cavity":
            b, f = _step_work(n, "tri", 8, 2 * n, 3)
        elif case["flow"] == "cube":
            b, f = _step_work(n, "tet", 8, 5 * n, 2)
        else:
            b, f = _step_work(n, "tet", 4 if case["fp32"] else 8, 3 * n, 2)
        return {"bytes": b, "flops": f}
    if case["kind"] == "si":
        N, _, nb = _sizes("quad", case["n"])
        its = 10 * case["n"]
        return {"bytes": its * 2 * (nb * 12 + N * 20), "flops": its * 4 * nb}
    b = f = 0
    for i in range(case["count"]):
        c = case["lo"] * (case["hi"] / case["lo"]) ** (i / max(case["count"] - 1, 1))
        sb, sf = _step_work(int(round(c)), "tet", 4, 3 * int(round(c)), 2)
        b, f = b + case["steps"] * sb, f + case["steps"] * sf
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "assemble":
        return {"rel": 1e-6, "max": 1e-4} if case["fp32"] else {"rel": 1e-12, "max": 1e-10}
    if case["kind"] == "step":
        return {"rel": 2e-6, "max": 1e-5}
    if case["kind"] == "si":
        return {"rel": 1e-11, "max": 1e-10}
    # solves to 1e-8: a pressure moves by up to 9e-4 when the tolerance goes to 1e-11
    return {"rel": 3e-3, "max": 1e-2}


# ------------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits, on whole element batches
# ------------------------------------------------------------------------------------------------
_X = 0.5773502691896257645091488


def _points(cell):
    """Reference points and weights of the order-2 rule and the point of the tau evaluation."""
    x = _X
    if cell == "tri":
        return [(0.5, 0.0), (0.5, 0.5), (0.0, 0.5)], [1 / 6.0] * 3, (1 / 3.0, 1 / 3.0)
    if cell == "tet":
        m = 0.13819660112501051517954131656
        q = 1.0 - 3.0 * m
        return [(m, m, m), (q, m, m), (m, q, m), (m, m, q)], [1 / 24.0] * 4, (0.25, 0.25, 0.25)
    if cell == "quad":
        return [(sx, sy) for sy in (-x, x) for sx in (-x, x)], [1.0] * 4, (0.0, 0.0)
    if cell == "hex":
        return ([(sx, sy, sz) for sz in (-x, x) for sy in (-x, x) for sx in (-x, x)], [1.0] * 8, (0.0, 0.0, 0.0))
    t = [(0.5, 0.0), (0.5, 0.5), (0.0, 0.5)]
    return [(a, b, z) for z in (x, -x) for a, b in t], [1 / 6.0] * 6, (1 / 3.0, 1 / 3.0, 0.0)


_HEX = [(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)]


def _shape(cell, xi):
    """Shape functions and their reference gradients (dim x k) at one point."""
    if cell in ("tri", "tet"):
        d = len(xi)
        N = [1.0 - sum(xi)] + list(xi)
        G = [[-1.0] + [1.0 if m == i else 0.0 for m in range(d)] for i in range(d)]
    elif cell in ("quad", "hex"):
        d = len(xi)
        corners = _HEX if d == 3 else [c[:2] for c in _HEX[:4]]
        N = [math.prod(0.5 * (1 + c[i] * xi[i]) for i in range(d)) for c in corners]
        G = [[0.5 * c[j] * math.prod(0.5 * (1 + c[i] * xi[i]) for i in range(d) if i != j) for c in corners]
             for j in range(d)]
    else:
        a, b, z = xi
        L, dL = [1 - a - b, a, b], [[-1.0, 1.0, 0.0], [-1.0, 0.0, 1.0]]
        lo, hi = 0.5 * (1 - z), 0.5 * (1 + z)
        N = [v * lo for v in L] + [v * hi for v in L]
        G = [[v * lo for v in dL[0]] + [v * hi for v in dL[0]], [v * lo for v in dL[1]] + [v * hi for v in dL[1]],
             [-0.5 * v for v in L] + [0.5 * v for v in L]]
    return torch.tensor(N, dtype=torch.float64, device=DEV), torch.tensor(G, dtype=torch.float64, device=DEV)


def _inverse(J):
    """Inverse and determinant of a batch of 2 x 2 or 3 x 3 matrices by cofactors."""
    if J.shape[-1] == 2:
        det = J[:, 0, 0] * J[:, 1, 1] - J[:, 0, 1] * J[:, 1, 0]
        adj = torch.stack([J[:, 1, 1], -J[:, 0, 1], -J[:, 1, 0], J[:, 0, 0]], 1).view(-1, 2, 2)
    else:
        r = [torch.linalg.cross(J[:, (i + 1) % 3], J[:, (i + 2) % 3]) for i in range(3)]
        det = (J[:, 0] * r[0]).sum(1)
        adj = torch.stack(r, 2)
    return adj / det[:, None, None], det


def _tau(cell, X, uc, nu, dt):
    """METRIC tau: (tau_ps = tau_su, tau_bulk)."""
    _, dN = _shape(cell, _points(cell)[2])
    Ji, _ = _inverse(dN @ X)
    g = Ji.transpose(1, 2) @ Ji
    ugu = ((uc[:, None, :] @ g)[:, 0] * uc).sum(1).abs()
    sq = (4.0 / dt ** 2 + ugu + 16.0 * nu ** 2 * (g * g).sum((1, 2))).sqrt()
    return 1.0 / sq, sq / torch.diagonal(g, dim1=1, dim2=2).sum(1)


def _tet_volume(X):
    """det J / 6 expanded in absolute coordinates, the volume that the specialised terms are defined with."""
    (x0, y0, z0), (x1, y1, z1), (x2, y2, z2), (x3, y3, z3) = (X[:, i].unbind(1) for i in range(4))
    return (x2*y1*z0 - x3*y1*z0 - x1*y2*z0 + x3*y2*z0 + x1*y3*z0 - x2*y3*z0 - x2*y0*z1 + x3*y0*z1 +
            x0*y2*z1 - x3*y2*z1 - x0*y3*z1 + x2*y3*z1 + x1*y0*z2 - x3*y0*z2 - x0*y1*z2 + x3*y1*z2 +
            x0*y3*z2 - x1*y3*z2 - x1*y0*z3 + x2*y0*z3 + x0*y1*z3 - x2*y1*z3 - x0*y2*z3 + x1*y2*z3) / 6.0


def _element_system(cell, spec, X, u, p, ua, nu, prm):
    """M = T/dt + theta A' and b = -A x of a batch of elements, rows and columns node-major."""
    rho, dt, theta = prm
    B, k, d = X.shape
    A = torch.zeros(B, k, d + 1, k, d + 1, dtype=torch.float64, device=DEV)
    T = torch.zeros_like(A)
    if spec:
        c = 1.0 / 6.0 if d == 2 else 1.0 / 12.0
        um, num = ua.mean(1), nu.mean(1).abs()
        Ji, det = _inverse(X[:, 1:] - X[:, :1])
        V = det / 2.0 if d == 2 else _tet_volume(X)
        G = torch.cat([-Ji.transpose(1, 2).sum(1, keepdim=True), Ji.transpose(1, 2)], 1)       # gradients
        n = G * (det / math.factorial(d) * d)[:, None, None]                                     # face normals
        ts, tb = _tau(cell, X, u.mean(1), num, dt)
        r = 1.0 / (d * d * V)
        # the reference's tetrahedron takes the y velocity for the z velocity in its skew terms
        us = um.clone()
        if d == 3:
            us[:, 2] = um[:, 1]
        un = (um[:, None] * n).sum(2)
        nn = n @ n.transpose(1, 2)
        cc = c + (ts * r)[:, None] * un
        diag = cc[:, :, None] * un[:, None, :] + (num * r)[:, None, None] * nn
        mass = (V / (12.0 if d == 2 else 20.0))[:, None, None] * (1 + torch.eye(k, dtype=torch.float64, device=DEV))
        tm = mass + (ts * c)[:, None, None] * un[:, :, None]
        for i in range(d):
            A[:, :, i, :, i] += diag
            T[:, :, i, :, i] += tm
            for j in range(d):
                A[:, :, i, :, j] += 0.5 * cc[:, :, None] * us[:, None, None, i] * n[:, None, :, j] + \
                    ((num / 3.0 + tb) * r)[:, None, None] * n[:, :, None, i] * n[:, None, :, j]
            A[:, :, i, :, d] += cc[:, :, None] * n[:, None, :, i] / rho
            A[:, :, d, :, i] += (ts * r)[:, None, None] * un[:, None, :] * n[:, :, None, i] + \
                (c + 0.5 * (ts * r)[:, None] * (us[:, None] * n).sum(2))[:, :, None] * n[:, None, :, i]
            T[:, :, d, :, i] += (ts * c)[:, None, None] * n[:, :, None, i]
        A[:, :, d, :, d] += (ts * r / rho)[:, None, None] * nn
    else:
        pts, wts, c0 = _points(cell)
        ts, tb = _tau(cell, X, torch.einsum("m,bmd->bd", _shape(cell, c0)[0], ua), nu.mean(1).abs(), dt)
        for xi, wq in zip(pts, wts):
            N, dN = _shape(cell, xi)
            Ji, det = _inverse(dN @ X)
            G = (Ji @ dN).transpose(1, 2)                                                        # B k d
            w = (wq * det)[:, None, None]
            uq, nuq = (N[None, :, None] * ua).sum(1), (N * nu).sum(1)
            L = (G * uq[:, None]).sum(2)
            SU = N + ts[:, None] * L
            gtg = G @ G.transpose(1, 2)
            Nk = N[None, None, :]
            for i in range(d):
                A[:, :, d, :, i] += w * ((N + 0.5 * ts[:, None] * L)[:, :, None] * G[:, None, :, i] +
                                         ts[:, None, None] * G[:, :, None, i] * L[:, None, :])
                A[:, :, i, :, i] += w * (nuq[:, None, None] * gtg + SU[:, :, None] * L[:, None, :])
                A[:, :, i, :, d] += w * SU[:, :, None] * G[:, None, :, i] / rho
                for j in range(d):
                    A[:, :, i, :, j] += w * (tb[:, None] * G[:, :, i] + 0.5 * uq[:, None, i] * SU)[:, :, None] * \
                        G[:, None, :, j]
                T[:, :, d, :, i] += w * ts[:, None, None] * G[:, :, None, i] * Nk
                T[:, :, i, :, i] += w * SU[:, :, None] * Nk
            A[:, :, d, :, d] += w * (ts[:, None, None] * gtg) / rho
    m = k * (d + 1)
    x = torch.cat([u, p[:, :, None]], 2).reshape(B, m, 1)
    b = -(A.view(B, m, m) @ x)[:, :, 0]
    A[:, :, :d] *= theta
    return (T / dt + A).view(B, m, m), b


class _Elements:
    """Element systems of a whole mesh in batches; `keep` holds the matrices for repeated products."""

    def __init__(self, cell, spec, f, keep):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
        self.conn = t(f.conn.astype(np.int64))
        self.neq = f.dim + 1
        self.dofs = f.n_nodes * self.neq
        self.args = cell, spec, t(f.coords), t(f.u0), t(f.p0), f.nu, (f.rho, f.dt, f.theta)
        self.step = 100000
        self.kept = [self.batch(i) for i in range(0, len(self.conn), self.step)] if keep else None

    def batch(self, i):
        cell, spec, X, u, p, nu, prm = self.args
        c = self.conn[i:i + self.step]
        M, b = _element_system(cell, spec, X[c], u[c], p[c], u[c], torch.full(c.shape, nu, dtype=torch.float64, device=DEV), prm)
        return (c[:, :, None] * self.neq + torch.arange(self.neq, device=DEV)).reshape(len(c), -1), M, b

    def batches(self):
        return self.kept if self.kept is not None else (self.batch(i) for i in range(0, len(self.conn), self.step))

    def products(self, *xs):
        """rhs, and A x for each x."""
        out = [torch.zeros(self.dofs, dtype=torch.float64, device=DEV) for _ in range(len(xs) + 1)]
        for at, M, b in self.batches():
            out[0].index_add_(0, at.view(-1), b.reshape(-1))
            for o, x in zip(out[1:], xs):
                o.index_add_(0, at.view(-1), (M @ x[at][:, :, None]).reshape(-1))
        return out

    def diagonal(self):
        d = torch.zeros(self.dofs, dtype=torch.float64, device=DEV)
        for at, M, _ in self.batches():
            d.index_add_(0, at.view(-1), torch.diagonal(M, dim1=1, dim2=2).reshape(-1))
        return d


def _solved_step(f, cell):
    """The fields after one implicit step: conditions eliminated, the system solved to 1e-14."""
    e = _Elements(cell, True, f, keep=True)
    first, last = {}, {}
    for _, nodes, spec in f.bc_regions:
        for node, c in zip(nodes.tolist(), f.coords[nodes]):
            for eq, v in sorted(spec.items()):
                new = float(v(c[None])[0]) if callable(v) else float(v)
                inc = new - (f.p0[node] if eq == f.dim else f.u0[node, eq])
                first.setdefault(node * e.neq + eq, inc)
                last[node * e.neq + eq] = inc
    at = torch.tensor(list(first), device=DEV)
    free = torch.ones(e.dofs, dtype=torch.float64, device=DEV)
    free[at] = 0.0
    vf = torch.zeros_like(free)
    vf[at] = torch.tensor(list(first.values()), dtype=torch.float64, device=DEV)
    b, moved = e.products(vf)
    b = free * (b - moved)
    D = torch.where(free > 0, e.diagonal(), torch.ones_like(free))
    op = lambda x: free * e.products(x)[1]  # noqa: E731
    x = torch.zeros_like(b)
    for _ in range(4):                       # BiCGStab, restarted on the true residual
        r = b - op(x)
        if r.norm() < 1e-14 * b.norm():
            break
        rh, pp, v, rho, al, om, goal = r.clone(), torch.zeros_like(r), torch.zeros_like(r), 1.0, 1.0, 1.0, 1e-14 * b.norm()
        for _ in range(1000):
            rho1 = torch.dot(rh, r)
            pp = r + (rho1 / rho * al / om) * (pp - om * v)
            rho = rho1
            ph = pp / D
            v = op(ph)
            al = rho / torch.dot(rh, v)
            s = r - al * v
            sh = s / D
            t = op(sh)
            om = torch.dot(t, s) / torch.dot(t, t)
            x = x + al * ph + om * sh
            r = s - om * t
            if not r.norm() > goal:
                break
    x[at] = torch.tensor([last[i] for i in first], dtype=torch.float64, device=DEV)
    x = x.view(-1, e.neq).cpu().numpy()
    return {"u": f.u0 + x[:, :f.dim], "p": f.p0 + x[:, f.dim]}


def exact(case, seed):
    if case["kind"] in ("si", "serve"):
        return None    # nested solves over several steps, no closed form: too long in plain torch
    f = _flow(case, seed)
    if case["kind"] == "step":
        return _solved_step(f, "tri" if case["flow"] == "cavity" else "tet")
    f.p0 = _pressure(f, seed)
    x = torch.from_numpy(_vector(f, seed, case["fp32"])).to(DEV).double()
    rhs, y = _Elements(case["cell"], case["spec"], f, keep=False).products(x)
    return {"y": y} if case["fp32"] else {"y": y, "rhs": rhs}
