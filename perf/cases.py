"""Workloads whose speed matters to a user of this package, as timed cases.

``listed()`` names them and says what each stands for; ``draw(rng)`` gives
another case of the same kinds and ranges; ``prepare`` builds what a program
holds before the call (mesh, plan or libCEED objects, device vectors), ``run``
is one pass through the public entry points, ``work`` what a pass cannot do
without and ``exact`` the same result from plain torch operations in 64 bits.

Kinds
  plan    HexOperator.apply on a plan built from a mesh (from_mesh)
  ceed    CeedOperatorApplyAdd / Apply of a gallery operator on geometric
          factors the caller holds in a CeedVector (the drop-in path)
  user    CeedOperatorApply of a user QFunction with two passive fields
          (restriction, basis, QFunction, transposes one after another)
  build   CeedOperatorApply of Poisson3DBuild: the geometric factors again,
          after the mesh has moved
  diag    HexOperator.assemble_diagonal on such a plan
  kappa   forward and backward of the variable-coefficient diffusion in torch
  cg      conjugate gradients on a plan

Meshes are boxes of nx * ny * nz trilinear hexes on the unit cube with the
interior vertices moved by up to 10% of the spacing; Q = p + 2 quadrature
points per direction (kappa: p + 1, as the benchmark's adjoint workload);
plans and operators run with the library's default launches.
"""

from __future__ import annotations

import functools
import math
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

import libceed_amd.ceed as libceed
from libceed_amd import HexMesh, ops
from libceed_amd.autograd import kappa_diffusion

QFUNCTIONS = Path(__file__).resolve().parent.parent / "tests" / "qfunctions" / "t-api.h"
KERNELS = {"mass": ops.QF_MASS, "poisson": ops.QF_DIFFUSION}
GALLERY = {("mass", 1): "MassApply", ("mass", 3): "Vector3MassApply",
           ("poisson", 1): "Poisson3DApply", ("poisson", 3): "Vector3Poisson3DApply"}
CHUNK = 1 << 22  # quadrature points at a time in exact()


def _case(name, kind, p, nx, ny=None, nz=None, form="poisson", ncomp=1, dtype="float64", **more):
    c = {"kind": kind, "p": p, "nx": nx, "ny": ny or nx, "nz": nz or nx, "form": form, "ncomp": ncomp, "dtype": dtype, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the coarsest level of a multigrid hierarchy or a unit test: one apply is launches and latency
        _case("apply_small_p2", "plan", 2, 6),
        # the benchmark's own workload: 8.1M DoFs, FP64 diffusion, order 4
        _case("apply_p4_8M", "plan", 4, 50),
        # low order on a box, where geometry weighs most per DoF
        _case("apply_p1_box", "plan", 1, 120, 100, 90),
        # high order, as few elements as the DoFs allow
        _case("apply_p7", "plan", 7, 19, 18, 21),
        # the inner operator of mixed-precision solves
        _case("apply_p6_f32", "plan", 6, 27, 24, 25, dtype="float32"),
        # drop-in libCEED use: gallery Poisson on a CeedVector of geometric factors
        _case("ceed_poisson_p4", "ceed", 4, 32),
        # three components at once (elasticity-like), summed into an existing vector
        _case("ceed_vector_p3", "ceed", 3, 31, 29, 27, ncomp=3, add=True),
        # a user QFunction of mass plus diffusion with two passive fields
        _case("user_staged_p3", "user", 3, 24, 22, 25),
        # geometric factors recomputed on a moved mesh
        _case("build_qdata_p4", "build", 4, 26, 25, 24),
        # Jacobi preconditioner set-up
        _case("diagonal_p5", "diag", 5, 22, 20, 19),
        # coefficient inversion: value and gradients in u and kappa
        _case("kappa_fwd_bwd_p4", "kappa", 4, 39),
        # 50 iterations of the solver on a mid-sized system
        _case("cg_p3", "cg", 3, 36, 33, 35, iterations=50),
    ]


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "ceed", "ceed", "user", "build", "diag", "kappa", "cg"])
    p = rng.randint(1, 8) if kind in ("plan", "ceed", "build") else rng.randint(2, 6)
    form = rng.choice(["poisson", "poisson", "mass"]) if kind in ("plan", "ceed", "diag") else "poisson"
    ncomp = rng.choice([1, 1, 3]) if kind in ("plan", "ceed") else 1
    dtype = rng.choice(["float64", "float64", "float32"]) if kind == "plan" else "float64"
    top = {"plan": 2.0e7, "ceed": 5.0e6, "user": 2.5e6, "build": 4.0e6, "diag": 2.5e6, "kappa": 7.0e6, "cg": 4.5e6}[kind]
    points = math.exp(rng.uniform(math.log(2.0e4), math.log(top / ncomp)))
    n = [max(2, round((points ** (1.0 / 3.0) / (p + 2)) * rng.uniform(0.85, 1.15))) for _ in range(3)]
    while n[0] * n[1] * n[2] * (p + 2) ** 3 > top / ncomp and max(n) > 2:
        n[n.index(max(n))] -= 1
    more = {"add": rng.random() < 0.5} if kind == "ceed" else {"iterations": 50} if kind == "cg" else {}
    return _case(None, kind, p, *n, form=form, ncomp=ncomp, dtype=dtype, **more)


# ---------------------------------------------------------------------------
# meshes and 1D bases


def _points(case):
    return case["p"] + (1 if case["kind"] == "kappa" else 2)


def _lex(n, p):
    """Element offsets [E, (p+1)^3] of the lexicographic numbering of a box of n elements of degree p."""
    P, M = p + 1, [k * p + 1 for k in n]
    ez, ey, ex = np.meshgrid(*(np.arange(k) for k in reversed(n)), indexing="ij")
    base = p * (ex + M[0] * (ey + M[1] * ez.astype(np.int64))).reshape(-1)
    i = np.arange(P)
    local = (i[None, None, :] + M[0] * (i[None, :, None] + M[1] * i[:, None, None])).reshape(-1)
    return (base[:, None] + local[None, :]).astype(np.int32)


@functools.lru_cache(maxsize=2)
def _topology(n, p):
    return _lex(n, p), _lex(n, 1)


def _mesh(case, seed):
    n, p = (case["nx"], case["ny"], case["nz"]), case["p"]
    rng = np.random.default_rng(seed)
    grid = np.meshgrid(*(np.linspace(0.0, 1.0, k + 1) for k in reversed(n)), indexing="ij")[::-1]  # x, y, z as [iz, iy, ix]
    coords = np.empty((3,) + grid[0].shape)
    for d in range(3):
        coords[d] = grid[d]
        coords[d][1:-1, 1:-1, 1:-1] += rng.uniform(-0.1 / n[d], 0.1 / n[d], tuple(k - 1 for k in reversed(n)))
    offsets, mesh_offsets = _topology(n, p)
    return HexMesh(n=n[0], p=p, num_elem=n[0] * n[1] * n[2], num_nodes=(n[0] * p + 1) * (n[1] * p + 1) * (n[2] * p + 1), offsets=offsets,
                   mesh_offsets=mesh_offsets, coords=coords.reshape(-1), num_vertices=coords[0].size)


@functools.lru_cache(maxsize=None)
def _basis(P, Q):
    """(B, G, w): Lagrange interpolation and derivative on P Gauss-Lobatto nodes at Q Gauss points, and the weights."""
    leg = np.polynomial.legendre.Legendre.basis(P - 1)
    nodes = np.concatenate([[-1.0], np.sort(leg.deriv().roots().real), [1.0]]) if P > 2 else np.array([-1.0, 1.0])
    x, w = np.polynomial.legendre.leggauss(Q)
    B, G = np.empty((Q, P)), np.zeros((Q, P))
    for a in range(P):
        others = [b for b in range(P) if b != a]
        B[:, a] = np.prod([(x - nodes[b]) / (nodes[a] - nodes[b]) for b in others], axis=0)
        for b in others:
            rest = [(x - nodes[c]) / (nodes[a] - nodes[c]) for c in others if c != b]
            G[:, a] += np.prod(rest, axis=0) / (nodes[a] - nodes[b]) if rest else 1.0 / (nodes[a] - nodes[b])
    return B, G, w


def _random(gen, n, dtype=torch.float64):
    return (torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) * 2 - 1).to(dtype)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 13)


# ---------------------------------------------------------------------------
# plain torch in 64 bits


def _along(x, M, axis):
    """Contract `axis` of x with the columns of M."""
    return torch.movedim(torch.tensordot(x, M, dims=([axis], [1])), -1, axis)


def _cube(x, Mx, My, Mz):
    """Tensor-product apply on [E, z, y, x]."""
    return _along(_along(_along(x, Mx, 3), My, 2), Mz, 1)


def _factors(mesh, Q, lo, hi, form):
    """Geometric factors of elements lo..hi: [E, 1 or 6, Q, Q, Q] (Voigt xx, yy, zz, yz, xz, xy)."""
    B, G, w = (torch.from_numpy(a).cuda() for a in _basis(2, Q))
    off = torch.from_numpy(mesh.mesh_offsets[lo:hi]).cuda().long()
    x = torch.from_numpy(mesh.coords.reshape(3, -1)).cuda()[:, off].reshape(3 * (hi - lo), 2, 2, 2)
    J = [d.reshape(3, hi - lo, Q, Q, Q) for d in (_cube(x, G, B, B), _cube(x, B, G, B), _cube(x, B, B, G))]  # J[d][c] = dx_c/dX_d
    A = [[J[(d + 1) % 3][(c + 1) % 3] * J[(d + 2) % 3][(c + 2) % 3] - J[(d + 1) % 3][(c + 2) % 3] * J[(d + 2) % 3][(c + 1) % 3] for c in range(3)]
         for d in range(3)]  # A[d][c] = det J * (dX_d/dx_c)
    det = sum(J[0][c] * A[0][c] for c in range(3))
    weight = w[:, None, None] * w[:, None] * w
    if form == "mass":
        return (weight * det)[:, None]
    s = weight / det
    return torch.stack([s * sum(A[a][c] * A[b][c] for c in range(3)) for a, b in ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))], 1)


def _chunks(mesh, Q):
    step = max(1, CHUNK // Q ** 3)
    for lo in range(0, mesh.num_elem, step):
        yield lo, min(mesh.num_elem, lo + step)


def _all_factors(mesh, Q, form):
    return torch.cat([_factors(mesh, Q, lo, hi, form).reshape(-1) for lo, hi in _chunks(mesh, Q)])


def _flux(S, g):
    """S grad, Voigt order."""
    return [S[:, 0] * g[0] + S[:, 5] * g[1] + S[:, 4] * g[2], S[:, 5] * g[0] + S[:, 1] * g[1] + S[:, 3] * g[2],
            S[:, 4] * g[0] + S[:, 3] * g[1] + S[:, 2] * g[2]]


def _plain_apply(mesh, Q, forms, u, factors=None, kappa=None, lam=None):
    """v = A u (component-major u); with lam, (A lam, grad lam . S grad u) of the kappa-weighted diffusion."""
    P = mesh.P
    B, G, _ = (torch.from_numpy(a).cuda() for a in _basis(P, Q))
    grads = ((G, B, B), (B, G, B), (B, B, G))
    N = mesh.num_nodes
    v = torch.zeros_like(u)
    dk = torch.empty(mesh.num_elem, Q, Q, Q, dtype=torch.float64, device="cuda") if lam is not None else None
    for lo, hi in _chunks(mesh, Q):
        off = torch.from_numpy(mesh.offsets[lo:hi]).cuda().long()
        for form in forms:
            S = factors[form].reshape(mesh.num_elem, -1, Q, Q, Q)[lo:hi] if factors else _factors(mesh, Q, lo, hi, form)
            for k in range(u.numel() // N):
                x = u[k * N:(k + 1) * N][off].reshape(-1, P, P, P)
                if form == "mass":
                    r = _cube(_cube(x, B, B, B) * S[:, 0], B.T, B.T, B.T)
                else:
                    if lam is not None:
                        gu = [_cube(x, *m) for m in grads]
                        x = lam[off].reshape(-1, P, P, P)
                    f = _flux(S, [_cube(x, *m) for m in grads])
                    if lam is not None:
                        dk[lo:hi] = sum(a * b for a, b in zip(f, gu))
                    if kappa is not None:
                        f = [a * kappa[lo:hi] for a in f]
                    r = sum(_cube(a, *(M.T for M in m)) for a, m in zip(f, grads))
                v[k * N:(k + 1) * N].index_add_(0, off.reshape(-1), r.reshape(-1))
    return v if lam is None else (v, dk.reshape(-1))


def _plain_diagonal(mesh, Q, form, factors):
    P = mesh.P
    B, G, _ = (torch.from_numpy(a).cuda() for a in _basis(P, Q))
    v = torch.zeros(mesh.num_nodes, dtype=torch.float64, device="cuda")
    terms = [(0, (B * B,) * 3, 1.0)] if form == "mass" else [
        (0, (G * G, B * B, B * B), 1.0), (1, (B * B, G * G, B * B), 1.0), (2, (B * B, B * B, G * G), 1.0),
        (3, (B * B, B * G, B * G), 2.0), (4, (B * G, B * B, B * G), 2.0), (5, (B * G, B * G, B * B), 2.0)]
    for lo, hi in _chunks(mesh, Q):
        S = factors.reshape(mesh.num_elem, -1, Q, Q, Q)[lo:hi]
        d = sum(f * _cube(S[:, k], *(M.T for M in m)) for k, m, f in terms)
        v.index_add_(0, torch.from_numpy(mesh.offsets[lo:hi]).cuda().long().reshape(-1), d.reshape(-1))
    return v


# ---------------------------------------------------------------------------
# states


def _inputs(case, seed):
    """The vectors a case starts from, made from the seed alone."""
    mesh, Q, gen = _mesh(case, seed), _points(case), _generator(seed)
    dtype = getattr(torch, case["dtype"])
    n = case["ncomp"] * mesh.num_nodes
    s = SimpleNamespace(mesh=mesh, Q=Q, u=_random(gen, n, dtype), v0=None, kappa=None, target=None)
    if case.get("add"):
        s.v0 = _random(gen, n)
    if case["kind"] == "cg":  # a right-hand side in the range of the pure Neumann operator
        s.u -= s.u.mean()
    if case["kind"] == "kappa":  # kappa = exp(g), |g| <= 0.5; a target field for the misfit
        s.kappa = torch.exp(0.5 * _random(gen, mesh.num_elem * Q ** 3))
        s.target = _random(gen, n) * 0.1
    return s


def _vector(ceed, t):
    v = ceed.Vector(t.numel())
    v.set_array(t.data_ptr(), memtype=libceed.MEM_DEVICE, cmode=libceed.USE_POINTER)
    return v


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, mesh, Q, ncomp, E = case["kind"], s.mesh, s.Q, case["ncomp"], s.mesh.num_elem
    s.kind, s.add, s.iterations = kind, case.get("add", False), case.get("iterations", 0)
    if kind in ("plan", "cg", "diag"):
        s.op = ops.HexOperator.from_mesh(KERNELS[case["form"]], mesh, Q=Q, num_comp=ncomp, dtype=s.u.dtype)
        s.v = torch.empty_like(s.u)
        if kind == "cg":
            s.solver = ops.CG(s.op)
        return s
    if kind == "kappa":
        s.op = ops.HexOperator.from_mesh(ops.QF_DIFFUSION_KAPPA, mesh, Q=Q)
        s.u.requires_grad_()
        s.kappa.requires_grad_()
        return s
    # libCEED objects on device arrays of the caller
    ceed = s.ceed = libceed.Ceed("/gpu/hip/mi355")
    P, N, nq = mesh.P, mesh.num_nodes, Q ** 3

    def strided(comps):
        return ceed.StridedElemRestriction(E, nq, comps, E * nq * comps, libceed.STRIDES_BACKEND)

    if kind == "build":
        s.x = torch.from_numpy(mesh.coords).cuda()
        s.v = torch.empty(E * 6 * nq, dtype=torch.float64, device="cuda")
        s.cx, s.cv = _vector(ceed, s.x), _vector(ceed, s.v)
        rstr = ceed.ElemRestriction(E, 8, 3, mesh.num_vertices, 3 * mesh.num_vertices, mesh.mesh_offsets)
        basis = ceed.BasisTensorH1Lagrange(3, 3, 2, Q, libceed.GAUSS)
        s.op = ceed.Operator(ceed.QFunctionByName("Poisson3DBuild"))
        s.op.set_field("dx", rstr, basis, libceed.VECTOR_ACTIVE)
        s.op.set_field("weights", libceed.ELEMRESTRICTION_NONE, basis, libceed.VECTOR_NONE)
        s.op.set_field("qdata", strided(6), libceed.BASIS_NONE, libceed.VECTOR_ACTIVE)
        return s
    rstr = ceed.ElemRestriction(E, P ** 3, ncomp, N, ncomp * N, mesh.offsets)
    basis = ceed.BasisTensorH1Lagrange(3, ncomp, P, Q, libceed.GAUSS)
    s.v = s.v0.clone() if s.add else torch.empty_like(s.u)
    s.cx, s.cv = _vector(ceed, s.u), _vector(ceed, s.v)
    s.factors = {f: _all_factors(mesh, Q, f) for f in (("mass", "poisson") if kind == "user" else (case["form"],))}
    s.cq = {f: _vector(ceed, t) for f, t in s.factors.items()}
    if kind == "user":
        qf = ceed.QFunction(1, None, f"{QFUNCTIONS}:user_mass_diffusion")
        qf.add_input("u", 1, libceed.EVAL_INTERP)
        qf.add_input("du", 3, libceed.EVAL_GRAD)
        qf.add_input("qm", 1, libceed.EVAL_NONE)
        qf.add_input("qd", 6, libceed.EVAL_NONE)
        qf.add_output("v", 1, libceed.EVAL_INTERP)
        qf.add_output("dv", 3, libceed.EVAL_GRAD)
        s.op = ceed.Operator(qf)
        for name in ("u", "du", "v", "dv"):
            s.op.set_field(name, rstr, basis, libceed.VECTOR_ACTIVE)
        s.op.set_field("qm", strided(1), libceed.BASIS_NONE, s.cq["mass"])
        s.op.set_field("qd", strided(6), libceed.BASIS_NONE, s.cq["poisson"])
        return s
    form = case["form"]
    names = ("u", "qdata", "v") if form == "mass" else ("du", "qdata", "dv")
    s.op = ceed.Operator(ceed.QFunctionByName(GALLERY[form, ncomp]))
    s.op.set_field(names[0], rstr, basis, libceed.VECTOR_ACTIVE)
    s.op.set_field(names[1], strided(1 if form == "mass" else 6), libceed.BASIS_NONE, s.cq[form])
    s.op.set_field(names[2], rstr, basis, libceed.VECTOR_ACTIVE)
    return s


def run(s):
    if s.kind == "plan":
        s.op.apply(s.u, s.v)
        return s.v
    if s.kind == "cg":
        s.v.zero_()
        stats = s.solver.solve(s.u, s.v, max_iter=s.iterations, rtol=1e-10, check_every=25)
        return s.v, stats.iterations
    if s.kind == "kappa":
        v = kappa_diffusion(s.u, s.kappa, s.op)
        misfit = 0.5 * (v - s.target).square().sum()
        return v.detach(), *torch.autograd.grad(misfit, (s.u, s.kappa))
    if s.kind == "diag":
        s.op.assemble_diagonal(s.v)
    elif s.add:
        s.op.apply_add(s.cx, s.cv)
    else:
        s.op.apply(s.cx, s.cv)
    return s.v


def work(case):
    p, Q, nc = case["p"], _points(case), case["ncomp"]
    P, n = p + 1, (case["nx"], case["ny"], case["nz"])
    E, N, V = math.prod(n), math.prod(k * p + 1 for k in n), math.prod(k + 1 for k in n)
    s, nq = (4 if case["dtype"] == "float32" else 8), Q ** 3
    mesh = 8 * 3 * V + 4 * 8 * E                   # coordinates and their offsets: the geometry of a plan built from a mesh
    vec, offs = s * nc * N, 4 * E * P ** 3
    interp = 2 * (Q * P ** 3 + Q * Q * P * P + nq * P)
    form = 2 * interp + (nq if case["form"] == "mass" else 12 * Q * nq + 15 * nq)
    kind = case["kind"]
    if kind == "plan":
        return {"bytes": 2 * vec + offs + mesh, "flops": E * nc * form}
    if kind == "cg":
        once = 10 * vec + offs + mesh              # apply, two dot products, three vector updates
        return {"bytes": case["iterations"] * once, "flops": case["iterations"] * (E * form + 10 * N)}
    if kind == "kappa":                            # forward: u, kappa, v; backward: target, u, v, kappa, du, dkappa
        return {"bytes": 7 * vec + 2 * (offs + mesh) + 8 * 3 * E * nq, "flops": E * (3 * form)}
    if kind == "build":
        return {"bytes": mesh + 8 * 6 * E * nq, "flops": E * (9 * 2 * (4 * Q * 2 + 2 * Q * Q * 2 + nq * 2) + 70 * nq)}
    if kind == "diag":
        return {"bytes": mesh + offs + vec, "flops": E * interp * (1 if case["form"] == "mass" else 6)}
    factors = 8 * E * nq * (1 if case["form"] == "mass" else 6)
    if kind == "user":
        return {"bytes": 2 * vec + offs + 8 * 7 * E * nq, "flops": E * (form + nq)}
    return {"bytes": (3 if case.get("add") else 2) * vec + offs + factors, "flops": E * nc * form}


def exact(case, seed):
    s = _inputs(case, seed)
    mesh, Q, kind, form = s.mesh, s.Q, case["kind"], case["form"]
    u = s.u.double()
    if kind == "plan":
        return _plain_apply(mesh, Q, (form,), u)
    if kind == "build":
        return _all_factors(mesh, Q, "poisson")
    if kind == "diag":
        return _plain_diagonal(mesh, Q, form, _all_factors(mesh, Q, form))
    if kind == "kappa":
        kappa = s.kappa.reshape(-1, Q, Q, Q)
        v = _plain_apply(mesh, Q, ("poisson",), u, kappa=kappa)
        return v, *_plain_apply(mesh, Q, ("poisson",), u, kappa=kappa, lam=v - s.target)
    forms = ("mass", "poisson") if kind == "user" else (form,)
    factors = {f: _all_factors(mesh, Q, f) for f in forms}
    if kind != "cg":
        v = _plain_apply(mesh, Q, forms, u, factors)
        return s.v0 + v if case.get("add") else v
    x, r = torch.zeros_like(u), u.clone()
    d, rr, bb, done = r.clone(), r @ r, u @ u, 0
    while done < case["iterations"] and rr > 1e-20 * bb:  # tested every 25 iterations
        for _ in range(25):
            Ad = _plain_apply(mesh, Q, forms, d, factors)
            alpha = rr / (d @ Ad)
            x, r = x + alpha * d, r - alpha * Ad
            new = r @ r
            d, rr = r + (new / rr) * d, new
        done += 25
    return x, None
