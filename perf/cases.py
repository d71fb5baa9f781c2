"""The work this framework is used for, as cases that can be timed and checked.

Every case goes through the package's public entry points: the LinearStatic
and StaticStructural drivers, hippcg solves and hipcsr products on assembled
matrices, the Newton update (return mapping with internal forces, then the
consistent tangent), the RVE batch, and the MisesMat surrogate's training
and use.  ``listed()`` names the standard cases, ``draw()`` gives more of
the same ranges, and ``exact()`` recomputes a case's outputs in 64 bits with
plain torch: its own shape functions, quadrature, return mapping, sparse
assembly and conjugate gradients.
"""
import ctypes
import math

import numpy as np
import torch

from oofem_amd import meshgen
from oofem_amd.drivers import LinearStaticProblem
from oofem_amd.hipfem import BatchedEvaluator, Context, DeviceVector, HipCSRSparseMtrx, HipPCGSolver, MisesSurrogate, lib
from oofem_amd.problem import StructuralProblem
from oofem_amd.rve import RVEBatch

HEX, TET, QUAD = meshgen.LSPACE, meshgen.LTRSPACE, meshgen.QSPACE
MISES = (210e3, 0.3, 250.0, 2e3)          # E, nu, sig0, H of the plasticity configurations
YIELD_STRAIN = MISES[2] / MISES[0]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a small LinearStatic problem from deck to reactions (the 10x10x40
        # cantilever): assembly, internal forces and about 500 short PCG iterations
        dict(name="static_small", kind="static", nx=10, ny=10, nz=40, tol=1e-10),
        # plain FP64 PCG on an elastic hexahedral cantilever (node-block
        # matrix) with no tile-aligned dimension
        dict(name="pcg_hex", kind="pcg", mesh="cantilever", nx=33, ny=31, nz=126, precision=0, tol=1e-10),
        # plain FP64 PCG on the plastic tangent of a tetrahedral block
        # (row-group matrix: the loaded face constrains one component)
        dict(name="pcg_tet", kind="pcg", mesh="tet", nx=35, ny=35, nz=41, precision=0, tol=1e-10),
        # mixed-precision PCG on the 3.2M-DOF cantilever, to the 1e-8 that
        # configuration is solved to
        dict(name="pcg_mixed_large", kind="pcg", mesh="cantilever", nx=64, ny=64, nz=256, precision=2, tol=1e-8),
        # one plastic load step of the hexahedral block through the C++
        # driver: initial guess, full Newton, one PCG solve per correction
        dict(name="newton_hex", kind="newton", nx=16, ny=16, nz=64, precision=0, tol=1e-8),
        # what a Newton iteration does beside the solve, on the 3.2M-DOF
        # plasticity block: internal forces with the return mapping, then
        # the consistent tangent
        dict(name="update_hex_large", kind="update", mesh="hex", nx=64, ny=64, nz=256, strain=1.5, step=0.3),
        # the same on the 2.4M-element tetrahedral block
        dict(name="update_tet_large", kind="update", mesh="tet", nx=70, ny=70, nz=82, strain=1.5, step=0.3),
        # elastic 20-node hexahedra (an RVE of odd size): forces and stiffness
        dict(name="update_quad", kind="update", mesh="quad", n=21, vf=0.3),
        # the matrix product alone on 256 million stored entries
        dict(name="spmv_large", kind="spmv", nx=64, ny=64, nz=256),
        # two-phase RVEs of uneven size and both element types, homogenised
        # by six unit-strain solves each
        dict(name="rve_batch", kind="rve", count=24, nmin=8, nmax=16, tol=1e-10),
        # Adam steps of the MisesMat surrogate (forward, backward, update)
        dict(name="surrogate_train", kind="train", samples=200000, batch=4096, steps=16),
        # internal forces with the surrogate switched on: classification,
        # BF16 inference, acceptance checks, plain fallback
        dict(name="update_surrogate", kind="surrogate", nx=32, ny=32, nz=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _block(rng, lo, hi, aspect=4.0):
    """An elongated block of nx x ny x nz cells, nx between lo and hi."""
    nx = _log_int(rng, lo, hi)
    ny = max(lo, min(hi, nx + rng.randint(-3, 3)))
    return dict(nx=nx, ny=ny, nz=max(lo, min(int(aspect * hi), int(aspect * nx) + rng.randint(-5, 5))))


def draw(rng):
    kind = rng.choice(["static", "pcg", "pcg_tet", "pcg_mixed", "newton", "update", "update_tet", "update_quad", "spmv",
                       "rve", "train", "surrogate"])
    if kind == "static":
        return dict(kind="static", tol=1e-10, **_block(rng, 3, 14))
    if kind == "pcg":
        return dict(kind="pcg", mesh="cantilever", precision=0, tol=1e-10, **_block(rng, 6, 40))
    if kind == "pcg_tet":
        return dict(kind="pcg", mesh="tet", precision=0, tol=1e-10, **_block(rng, 8, 56, 1.2))
    if kind == "pcg_mixed":
        return dict(kind="pcg", mesh="cantilever", precision=2, tol=1e-8, **_block(rng, 10, 62))
    if kind == "newton":
        return dict(kind="newton", precision=rng.choice([0, 2]), tol=1e-8, **_block(rng, 4, 16))
    if kind == "update":
        return dict(kind="update", mesh="hex", strain=round(rng.uniform(0.8, 2.5), 2), step=round(rng.uniform(0.1, 0.5), 2),
                    **_block(rng, 6, 62))
    if kind == "update_tet":
        return dict(kind="update", mesh="tet", strain=round(rng.uniform(0.8, 2.5), 2), step=round(rng.uniform(0.1, 0.5), 2),
                    **_block(rng, 6, 68, 1.2))
    if kind == "update_quad":
        return dict(kind="update", mesh="quad", n=rng.randint(8, 32), vf=round(rng.uniform(0.1, 0.4), 2))
    if kind == "spmv":
        return dict(kind="spmv", **_block(rng, 8, 62))
    if kind == "rve":
        lo = rng.randint(4, 12)
        return dict(kind="rve", count=_log_int(rng, 4, 32), nmin=lo, nmax=lo + rng.randint(1, 6), tol=1e-10)
    if kind == "train":
        return dict(kind="train", samples=_log_int(rng, 50000, 1000000), batch=_log_int(rng, 500, 8192),
                    steps=rng.randint(8, 20))
    return dict(kind="surrogate", **_block(rng, 8, 40))


# --------------------------------------------------------------------- inputs
def _deck(case, seed):
    if case["kind"] in ("static", "spmv") or case.get("mesh") == "cantilever":
        return meshgen.config1(case["nx"], case["ny"], case["nz"], seed=seed)
    if case.get("mesh") == "tet":
        return meshgen.config2(case["nx"], case["ny"], case["nz"], seed=seed)
    if case.get("mesh") == "quad":
        return meshgen.rve(case["n"], QUAD, case["vf"], seed)
    return meshgen.config3(case["nx"], case["ny"], case["nz"], seed=seed)


def _field(d, strain, seed):
    """A displacement state of the ramped block, in yield strains: uniaxial
    extension with nodal noise of a tenth of a yield strain per cell; free and
    prescribed values."""
    z = d.coords[:, 2]
    zmax = z.max()
    h = zmax / d.meta["nz"]
    u = 0.1 * YIELD_STRAIN * h * np.random.default_rng(seed).standard_normal((d.nnode, 3))
    u[:, 2] += strain * YIELD_STRAIN * z
    up = d.prescribed_values(strain * YIELD_STRAIN * zmax / d.meta["u_end"])
    uf = np.zeros(d.neq)
    m = d.eqn > 0
    uf[d.eqn[m] - 1] = u[m]
    return uf, up


def _quad_field(d, seed):
    """Affine boundary values of a seeded macro strain of 1e-3 and a noisy
    affine field inside."""
    rng = np.random.default_rng(seed)
    e = rng.standard_normal(6)
    e *= 1e-3 / np.linalg.norm(e)
    u = (d.coords - 0.5) @ meshgen.macro_gradient(e).T + 1e-5 * rng.standard_normal(d.coords.shape)
    uf = np.zeros(d.neq)
    m = d.eqn > 0
    uf[d.eqn[m] - 1] = u[m]
    return uf, meshgen.affine_values(d, e)


def _states(case, d, seed):
    """(committed, current) displacement states of an update-like case."""
    if d.etype == QUAD:
        return None, _quad_field(d, seed + 1)
    s = case.get("strain", 1.5)
    return _field(d, s, seed + 1), _field(d, s + case.get("step", 0.3), seed + 2)


def _specs(case, seed):
    return meshgen.config4(case["count"], seed=seed, nmin=case["nmin"], nmax=case["nmax"])[0]


# --------------------------------------------------------------------- passes
_context = []


def _ctx():
    """The program's one GPU context."""
    if not _context:
        _context.append(Context(0))
    return _context[0]


class _View:
    """Device memory of an object of the package, as torch takes it (the
    tensor made from it keeps the object alive)."""

    def __init__(self, owner, addr, n):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(addr, False), version=2)


def _tensor(owner, addr, n):
    return torch.as_tensor(_View(owner, addr, n), device="cuda") if n else torch.zeros(0, dtype=torch.float64)


def _values(K):
    p = ctypes.c_void_p()
    lib().hipcsr_device_arrays(K.h, None, None, ctypes.byref(p))
    return _tensor(K, p.value, K.nnz())


class _Batch:
    def __init__(self, specs, tol):
        self.b = RVEBatch(_ctx(), specs)
        self.b.set_options(tol=tol)

    def __del__(self):
        self.b.close()


def _evaluator(case, seed):
    """Mesh, evaluator, matrix pattern and the device vectors of an update."""
    ctx = _ctx()
    d = _deck(case, seed)
    ev = BatchedEvaluator(ctx, d)
    K = HipCSRSparseMtrx(ctx)
    ev.build_structure(K)
    before, (uf, up) = _states(case, d, seed)
    if before is not None:
        ev.internal_forces(*before, update_state=True)
        ev.commit()
    v = [DeviceVector(ctx, n, x) for n, x in ((d.neq, uf), (d.npeq, up), (d.neq, None), (d.npeq, None))]
    return dict(d=d, ev=ev, K=K, u=v[0], up=v[1], f=v[2], fp=v[3], state=(uf, up))


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    if kind == "static":
        return dict(kind=kind, p=LinearStaticProblem(ctx, _deck(case, seed), lstol=case["tol"]))
    if kind == "newton":
        d = _deck(case, seed)
        p = StructuralProblem(d, lstol=case["tol"], mixed=case["precision"])
        p.set_load(None)
        p.set_prescribed(d.prescribed_values(5 / 20))   # the load steps up to the first plastic one
        if p.nonlinear_step()["status"] != 1:
            raise RuntimeError("the first load step did not converge")
        p.update()
        p.save_converged()
        p.set_prescribed(d.prescribed_values(6 / 20))
        return dict(kind=kind, p=p)
    if kind == "rve":
        return dict(kind=kind, p=_Batch(_specs(case, seed), case["tol"]))
    if kind == "train":
        net = MisesSurrogate(ctx, *MISES, seed=seed)
        net.generate(case["samples"], seed=seed + 1)
        return dict(kind=kind, p=net, batch=case["batch"], steps=case["steps"], seed=seed + 2)
    if kind in ("pcg", "spmv"):
        if case.get("mesh") == "tet":
            s = _evaluator(case, seed)
            d, ev, K = s["d"], s["ev"], s["K"]
            ev.internal_forces(*s["state"], update_state=True)
            ev.assemble_stiffness(K, tangent=True)
            b = -ev.tangent_product(None, d.prescribed_values(1 / 20))[0]   # the next load step's initial guess
        else:
            d = _deck(case, seed)
            ev = BatchedEvaluator(ctx, d)
            K = HipCSRSparseMtrx(ctx)
            ev.build_structure(K)
            ev.assemble_stiffness(K)
            b = np.random.default_rng(seed).standard_normal(d.neq) if kind == "spmv" else d.external_load()[0]
        x, y = DeviceVector(ctx, d.neq, b), DeviceVector(ctx, d.neq)
        solver = HipPCGSolver(ctx, lstol=case["tol"], lsiter=100000, precision=case["precision"]) if kind == "pcg" else None
        return dict(kind=kind, ev=ev, K=K, solver=solver, b=x, x=y, n=d.neq)
    s = dict(_evaluator(case, seed), kind=kind)
    if kind == "surrogate":
        s["net"] = MisesSurrogate(ctx, *MISES, seed=seed)
        s["net"].generate(100000, seed=seed + 1)
        s["net"].train(200, seed=seed + 2)
        s["ev"].set_surrogate(s["net"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "static":
        r = s["p"].solve()
        return r["u"], r["reactions"]
    if kind == "newton":
        s["p"].restart_step()
        if s["p"].nonlinear_step()["status"] != 1:
            raise RuntimeError("the load step did not converge")
        return s["p"].solution(), s["p"].reactions()
    if kind == "rve":
        return s["p"].b.run()["C"]
    if kind == "train":
        loss = s["p"].train(s["steps"], batch=s["batch"], seed=s["seed"])
        return s["p"].params(), loss
    if kind == "pcg":
        s["x"].fill(0.0)
        if s["solver"].solve_dev(s["K"], s["b"].addr, s["x"].addr)[0] != 1:
            raise RuntimeError("the solve did not converge")
        return _tensor(s["x"], s["x"].addr, s["n"])
    if kind == "spmv":
        s["K"].times_dev(s["b"].addr, s["x"].addr)
        return _tensor(s["x"], s["x"].addr, s["n"])
    d = s["d"]
    ebe = s["ev"].internal_forces_dev(s["u"].addr, s["up"].addr, s["f"].addr, s["fp"].addr,
                                      update_state=kind == "update", want_ebe=True)
    out = [_tensor(s["f"], s["f"].addr, d.neq), _tensor(s["fp"], s["fp"].addr, d.npeq), ebe]
    if kind == "update":
        s["ev"].assemble_stiffness(s["K"], tangent=True)
        out.append(_values(s["K"]))
    return out


# ----------------------------------------------------------------------- work
def _mesh_counts(case):
    """Elements, nodes, stored entries, Gauss points and nodes per element."""
    if case.get("mesh") == "quad":
        n = case["n"]
        nodes = (n + 1) ** 3 + 3 * n * (n + 1) ** 2
        return n ** 3, nodes, 9 * 58 * nodes, 27, 20
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cells, nodes = nx * ny * nz, (nx + 1) * (ny + 1) * (nz + 1)
    if case.get("mesh") == "tet":
        return 6 * cells, nodes, 9 * 15 * nodes, 1, 4
    return cells, nodes, 9 * (3 * nx + 1) * (3 * ny + 1) * (3 * nz + 1), 8, 8


def _iteration(nnz, n, precision, elements):
    """Bytes and flops of one Jacobi-PCG iteration: the operator read once
    (values with a column index per 3x3 block, or the element data of the
    FP32 element-by-element form), every vector read and written once."""
    if precision:
        return elements * 120 + 52 * n, elements * 3300 + 12 * n
    return nnz * (8 + 4 / 9) + 72 * n, 2 * nnz + 12 * n


def _update_work(case, tangent):
    ne, nn, nnz, ngp, nen = _mesh_counts(case)
    plastic = case.get("mesh") != "quad"
    by = ne * 4 * (nen + 1) + nn * (24 + 12 + 24 + 24) + ne * ngp * 8 * ((7 if plastic else 0) + (25 if tangent and plastic else 12 if tangent else 0))
    fl = ne * ngp * (nen * 90 + 200)
    if tangent:
        by += 8 * nnz
        fl += ne * ngp * nen * (nen + 1) / 2 * 9 * 6
    return by, fl


def work(case):
    kind = case["kind"]
    if kind == "train":
        p = 13 * 128 + 2 * 128 * 128 + 128 * 27
        return dict(bytes=case["steps"] * (28 * p + 4 * 40 * case["batch"]), flops=case["steps"] * 6.0 * p * case["batch"])
    if kind == "rve":
        by = fl = 0.0
        n = 0.5 * (case["nmin"] + case["nmax"])
        for share, nodes, width in ((0.7, (n - 1) ** 3, 27), (0.3, (n - 1) ** 3 + 3 * n * (n - 1) ** 2, 58)):
            it = 12.0 * n * (2 if width > 27 else 1)     # FP32 values, six columns at once
            by += share * it * (nodes * width * (36 + 4) + 3 * nodes * 6 * 40)
            fl += share * it * 12 * 9 * nodes * width
        return dict(bytes=case["count"] * by, flops=case["count"] * fl)
    ne, nn, nnz, ngp, nen = _mesh_counts(case)
    n = 3 * nn
    if kind == "spmv":
        return dict(bytes=nnz * (8 + 4 / 9) + 16 * n, flops=2.0 * nnz)
    if kind in ("update", "surrogate"):
        by, fl = _update_work(case, kind == "update")
        if kind == "surrogate":
            fl += ne * ngp * 2.0 * (13 * 128 + 2 * 128 * 128 + 128 * 27)
        return dict(bytes=by, flops=fl)
    by, fl = _iteration(nnz, n, case.get("precision", 0), ne)
    if kind == "pcg":       # iterations grow with the cells along the block
        it = case["nz"] * (19.0 if case.get("mesh") == "tet" else 12.0)
        return dict(bytes=it * by, flops=it * fl)
    ub, uf = _update_work(case, True)
    if kind == "static":
        return dict(bytes=case["nz"] * 12.0 * by + ub, flops=case["nz"] * 12.0 * fl + uf)
    it = 8 * case["nz"] * 12.0     # newton: about seven corrections and the initial guess
    return dict(bytes=it * by + 8 * ub, flops=it * fl + 8 * uf)


# --------------------------------------------------------------- 64-bit values
# Local node positions of the brick elements: xi, eta, zeta of the eight
# corners, then the mid-edge nodes of the 20-node brick.
_CORNERS = [(-1, -1, 1), (-1, 1, 1), (1, 1, 1), (1, -1, 1), (-1, -1, -1), (-1, 1, -1), (1, 1, -1), (1, -1, -1)]
_EDGES = [(-1, 0, 1), (0, 1, 1), (1, 0, 1), (0, -1, 1), (-1, 0, -1), (0, 1, -1), (1, 0, -1), (0, -1, -1),
          (-1, -1, 0), (-1, 1, 0), (1, 1, 0), (1, -1, 0)]


def _rule(etype):
    """Shape-function derivatives (points, nodes, 3) and weights; the bricks'
    points with zeta fastest, as the state orders them (it is not compared)."""
    if etype == TET:
        return torch.tensor([[[1.0, 0, 0], [0, 1, 0], [0, 0, 1], [-1, -1, -1]]], dtype=torch.float64), torch.tensor([1 / 6.0], dtype=torch.float64)
    x, w = (np.array([-1, 1]) / math.sqrt(3), np.ones(2)) if etype == HEX else (np.array([-1, 0, 1]) * math.sqrt(0.6), np.array([5, 8, 5]) / 9)
    pts = torch.tensor([(a, b, c) for a in x for b in x for c in x], dtype=torch.float64, requires_grad=True)
    wts = torch.tensor([a * b * c for a in w for b in w for c in w], dtype=torch.float64)
    cols = []
    for p in _CORNERS + (_EDGES if etype == QUAD else []):
        g = [1 + p[j] * pts[:, j] if p[j] else 1 - pts[:, j] ** 2 for j in range(3)]
        N = g[0] * g[1] * g[2] / (4 if 0 in p else 8)
        if etype == QUAD and 0 not in p:
            N = N * (p[0] * pts[:, 0] + p[1] * pts[:, 1] + p[2] * pts[:, 2] - 2)
        cols.append(torch.autograd.grad(N.sum(), pts, retain_graph=True)[0])
    return torch.stack(cols, 1), wts


class _Fem:
    """Plain torch finite elements of one deck, element batches at a time."""

    def __init__(self, d, device="cuda"):
        self.d = d
        t = lambda a, k: torch.as_tensor(np.ascontiguousarray(a), dtype=k, device=device)  # noqa: E731
        self.conn, self.X = t(d.conn, torch.int64), t(d.coords, torch.float64)
        self.dN, self.w = (a.to(device) for a in _rule(d.etype))
        eq = t(d.eqn, torch.int64)
        self.eq = torch.where(eq > 0, eq - 1, d.neq - eq - 1)[self.conn].reshape(d.nelem, -1)   # free, then prescribed
        self.n = d.neq + d.npeq
        mat = t(d.mat, torch.float64)[t(d.emat, torch.int64)]
        self.mises = bool(d.mat[0, 0] == meshgen.MAT_MISES)
        self.E, self.nu = mat[:, 1], mat[:, 2]
        self.G, self.B = self.E / (2 * (1 + self.nu)), self.E / (3 * (1 - 2 * self.nu))
        ngp = self.w.numel()
        self.ep = torch.zeros(d.nelem, ngp, 6, dtype=torch.float64, device=device) if self.mises else None
        self.kappa = torch.zeros(d.nelem, ngp, dtype=torch.float64, device=device) if self.mises else None
        self.step = max(1, int(4e7 / (ngp * 18 * self.conn.shape[1])))

    def vector(self, uf, up):
        dev = self.X.device
        return torch.cat([torch.as_tensor(uf, dtype=torch.float64).to(dev), torch.as_tensor(up, dtype=torch.float64).to(dev)])

    def _chunk(self, a):
        """Strain matrices (elements, points, 6, dofs) and volumes of a batch."""
        s = slice(a, min(a + self.step, self.d.nelem))
        J = torch.einsum("eni,gnj->egij", self.X[self.conn[s]], self.dN)
        g = torch.einsum("gnk,egkj->egnj", self.dN, torch.linalg.inv(J))
        B = torch.zeros(*g.shape[:2], 6, g.shape[2], 3, dtype=torch.float64, device=g.device)
        for r, pairs in enumerate([[(0, 0)], [(1, 1)], [(2, 2)], [(1, 2), (2, 1)], [(0, 2), (2, 0)], [(0, 1), (1, 0)]]):
            for c, j in pairs:
                B[:, :, r, :, c] = g[..., j]
        return s, B.flatten(3), torch.linalg.det(J).abs() * self.w

    def _material(self, s, eps, commit):
        """Stress and consistent tangent of the isotropic or J2 material."""
        G, K = self.G[s, None], self.B[s, None]
        dev = torch.zeros(6, 6, dtype=torch.float64, device=eps.device)
        dev[:3, :3] = -1 / 3
        dev += torch.diag(torch.tensor([1.0, 1, 1, 0.5, 0.5, 0.5], dtype=torch.float64, device=eps.device))
        one = torch.tensor([1.0, 1, 1, 0, 0, 0], dtype=torch.float64, device=eps.device)
        el = eps - self.ep[s] if self.mises else eps
        t = 2 * G[..., None] * (el @ dev)
        p = (K * el[..., :3].sum(-1))[..., None] * one
        D = 2 * G[..., None, None] * dev + K[..., None, None] * torch.outer(one, one)
        if not self.mises:
            return t + p, D
        sig0, H = MISES[2], MISES[3]
        norm = ((t * t) @ torch.tensor([1.0, 1, 1, 2, 2, 2], dtype=torch.float64, device=eps.device)).sqrt()
        sy = sig0 + H * self.kappa[s]
        dk = ((math.sqrt(1.5) * norm - sy) / (H + 3 * G)).clamp(min=0)
        on, safe = (dk > 0).double(), torch.where(norm > 0, norm, torch.ones_like(norm))
        f = -2 * math.sqrt(6) * G * G / safe
        sig = t * (1 - math.sqrt(6) * G * dk / safe)[..., None] + p
        D = D + (on * f * sy / ((H + 3 * G) * safe ** 2))[..., None, None] * (t[..., :, None] * t[..., None, :]) + (f * dk)[..., None, None] * dev
        if commit:
            self.ep[s] += (math.sqrt(1.5) * dk / safe)[..., None] * t * torch.tensor([1.0, 1, 1, 2, 2, 2], dtype=torch.float64, device=eps.device)
            self.kappa[s] += dk
        return sig, D

    def evaluate(self, u, matrix=True, commit=False):
        """Forces at every dof, squared element forces per component, and the
        sparse matrix over all dofs."""
        f, ebe = torch.zeros(self.n, dtype=torch.float64, device=u.device), torch.zeros(3, dtype=torch.float64, device=u.device)
        parts = []
        for a in range(0, self.d.nelem, self.step):
            s, B, dV = self._chunk(a)
            sig, D = self._material(s, torch.einsum("egrk,ek->egr", B, u[self.eq[s]]), commit)
            fe = torch.einsum("egrk,egr,eg->ek", B, sig, dV)
            f.index_add_(0, self.eq[s].reshape(-1), fe.reshape(-1))
            ebe += (fe * fe).reshape(-1, 3).sum(0)
            if matrix:
                Bf = B.flatten(1, 2)
                DB = torch.matmul(D * dV[..., None, None], B).flatten(1, 2)
                parts.append(torch.matmul(Bf.transpose(1, 2).contiguous(), DB))
        return f, ebe, self._csr(torch.cat(parts)) if matrix else None

    def _csr(self, Ke):
        n, k = self.n, self.eq.shape[1]
        i = self.eq[:, :, None].expand(-1, -1, k).reshape(-1)
        j = self.eq[:, None, :].expand(-1, k, -1).reshape(-1)
        free = (i < self.d.neq) if self.d.neq else i < n
        i, j, v = i[free], j[free], Ke.reshape(-1)[free]
        return torch.sparse_coo_tensor(torch.stack([i, j]), v, (self.d.neq, n)).coalesce()

    def split(self, A):
        """(free-free CSR, free-prescribed COO) of the free rows."""
        ij, v, n = A.indices(), A.values(), self.d.neq
        ff = ij[1] < n
        row = torch.zeros(n + 1, dtype=torch.int64, device=v.device)
        row[1:] = torch.bincount(ij[0, ff], minlength=n).cumsum(0)
        return torch.sparse_csr_tensor(row, ij[1, ff], v[ff], (n, n)), torch.sparse_coo_tensor(ij[:, ~ff] - torch.tensor([[0], [n]], device=v.device), v[~ff], (n, self.d.npeq))


def _diagonal(A):
    rows = torch.repeat_interleave(torch.arange(A.shape[0], device=A.device), A.crow_indices().diff())
    on = rows == A.col_indices()
    return A.values()[on]


def _solve(A, b, tol=1e-13, maxit=20000):
    """Jacobi conjugate gradients on columns, to (near) the attainable accuracy."""
    D = _diagonal(A)[:, None]
    b = b.reshape(b.shape[0], -1)
    x, r = torch.zeros_like(b), b.clone()
    stop = tol * b.norm(dim=0).clamp(min=1e-300)
    p = torch.zeros_like(b)
    rho = torch.ones(b.shape[1], dtype=b.dtype, device=b.device)
    for it in range(maxit):
        z = r / D
        new = (r * z).sum(0)
        p = z + (new / rho if it else 0.0) * p
        q = torch.sparse.mm(A, p) if p.shape[1] > 1 else (A @ p[:, 0])[:, None]
        a = new / (p * q).sum(0).clamp(min=1e-300)
        x, r, rho = x + a * p, r - a * q, new.clamp(min=1e-300)
        if it % 50 == 49 and bool((r.norm(dim=0) <= stop).all()):
            break
    return x


def _exact_newton(d):
    """Two load steps of the block (a quarter of the end displacement, then
    6/20 of it), each from the tangent's prediction; displacements and
    reactions of the second."""
    F = _Fem(d)
    u = F.vector(np.zeros(d.neq), np.zeros(d.npeq))
    for frac in (5 / 20, 6 / 20):
        up = F.vector(np.zeros(0), d.prescribed_values(frac))
        Aff, Afp = F.split(F.evaluate(u)[2])
        du = _solve(Aff, -torch.sparse.mm(Afp, (up - u[d.neq:])[:, None]))[:, 0]
        u = torch.cat([u[:d.neq] + du, up])
        for _ in range(30):
            f, _, A = F.evaluate(u)
            if float(f[:d.neq].norm()) <= 1e-13 * float(f.norm()):
                break
            u[:d.neq] -= _solve(F.split(A)[0], f[:d.neq])[:, 0]
        f = F.evaluate(u, matrix=False, commit=True)[0]
    return u[:d.neq], f[d.neq:]


def _exact_rve(spec):
    """Homogenised stiffness: the energies of the six unit-strain fields."""
    d = meshgen.rve(*spec)
    F = _Fem(d)
    Aff, Afp = F.split(F.evaluate(F.vector(np.zeros(d.neq), np.zeros(d.npeq)))[2])
    up = torch.as_tensor(np.stack([meshgen.affine_values(d, e) for e in np.eye(6)], 1), device="cuda")
    uf = _solve(Aff, -torch.sparse.mm(Afp, up))
    C = torch.stack([F.evaluate(torch.cat([uf[:, k], up[:, k]]), matrix=False)[0][d.neq:] @ up for k in range(6)], 1)
    return C.cpu().numpy()


def _mix(x):
    x = (x + np.uint64(0x9E3779B97F4A7C15)).astype(np.uint64)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _exact_train(case, seed):
    """The same Adam steps in 64 bits on the same batches (drawn by the
    documented counter hash)."""
    net = MisesSurrogate(_ctx(), *MISES, seed=seed)
    net.generate(case["samples"], seed=seed + 1)
    X, Y = (torch.as_tensor(a, dtype=torch.float64) for a in net.samples(0, case["samples"]))
    p = torch.as_tensor(net.params(), dtype=torch.float64)
    sizes = [(128, 13), (128,), (128, 128), (128,), (128, 128), (128,), (27, 128), (27,)]
    m, v, loss = torch.zeros_like(p), torch.zeros_like(p), None
    for it in range(case["steps"]):
        with np.errstate(over="ignore"):
            h = _mix(np.uint64(seed + 2) ^ _mix(np.uint64(it) * np.uint64(0x9E3779B97F4A7C15) + np.arange(case["batch"], dtype=np.uint64)))
        rows = torch.as_tensor((h % np.uint64(case["samples"])).astype(np.int64))
        q = p.clone().requires_grad_(True)
        W, o = [], 0
        for s in sizes:
            k = math.prod(s)
            W.append(q[o:o + k].reshape(s))
            o += k
        a = X[rows]
        for L in range(3):
            a = torch.nn.functional.silu(a @ W[2 * L].T + W[2 * L + 1])
        loss = ((a @ W[6].T + W[7] - Y[rows]) ** 2).mean()
        g = torch.autograd.grad(loss, q)[0]
        lr = 1e-5 + (1e-3 - 1e-5) * 0.5 * (1 + math.cos(math.pi * it / max(1, case["steps"])))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1 - 0.9 ** (it + 1))) / ((v / (1 - 0.999 ** (it + 1))).sqrt() + 1e-8)
    return p.numpy(), float(loss)


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "rve":
        return np.stack([_exact_rve(s) for s in _specs(case, seed)])
    d = _deck(case, seed)
    if kind == "newton":
        return _exact_newton(d)
    F = _Fem(d)
    if kind in ("update", "surrogate"):
        before, now = _states(case, d, seed)
        if before is not None:
            F.evaluate(F.vector(*before), matrix=False, commit=True)
        f, ebe, A = F.evaluate(F.vector(*now), matrix=kind == "update")
        out = [f[:d.neq], f[d.neq:], ebe]
        return out + [F.split(A)[0].values()] if kind == "update" else out
    if case.get("mesh") == "tet":
        before, now = _states(case, d, seed)
        F.evaluate(F.vector(*before), matrix=False, commit=True)
        Aff, Afp = F.split(F.evaluate(F.vector(*now))[2])
        b = -torch.sparse.mm(Afp, torch.as_tensor(d.prescribed_values(1 / 20), device="cuda")[:, None])
    else:
        Aff, _ = F.split(F.evaluate(F.vector(np.zeros(d.neq), np.zeros(d.npeq)))[2])
        if kind == "spmv":
            return Aff @ torch.as_tensor(np.random.default_rng(seed).standard_normal(d.neq), device="cuda")
        b = torch.as_tensor(d.external_load()[0], device="cuda")
    x = _solve(Aff, b)[:, 0]
    if kind == "static":
        fp = F.evaluate(torch.cat([x, torch.zeros(d.npeq, dtype=x.dtype, device=x.device)]), matrix=False)[0][d.neq:]
        return x, fp - torch.as_tensor(d.external_load()[1], device="cuda")
    return x
