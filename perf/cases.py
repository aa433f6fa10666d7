"""Workloads of the assembly + PCG path, for timing and for checking results.

Every case is one call sequence of a program that uses the library through
``lehrfempp_amd.capi``: the mesh, the plan and the device vectors are what such
a program keeps (``prepare``), the assembly, the solve and the download of the
result are the pass (``run``).  Meshes are rectangles of triangles; the DOF
numbering of the P3 space is vertices, then two DOFs an edge, then one a cell.

Kinds of cases
  p1        reaction-diffusion, P1, a = exp(theta) per cell, f = sin sin, zero
            Dirichlet data: assembly and one Jacobi-PCG solve
  demo      the constant-coefficient Poisson-like demo problem on a small mesh
  flipped   P1 on jittered meshes whose squares are cut along a random
            diagonal (no band structure)
  p3        P3 on jittered meshes, source and coefficient per cell
  batch_p1  many P1 problems of uneven sizes, assembled and solved together
  batch_p3  the same for P3
  adjoint   forward solve, adjoint solve and the gradient by cell coefficient
  fkpp      Fisher/KPP time stepping (Strang splitting), with or without the
            nonlocal boundary terms
  handoff   assembly with Robin and Neumann boundary terms, the matrix and the
            load vector handed to the host for a direct solver there
"""
from __future__ import annotations

import math

import numpy as np
import torch

from lehrfempp_amd import capi

MODES = {"fp64": capi.PCG_FP64, "mixed": capi.PCG_MIXED,
         "mixed_matrix": capi.PCG_MIXED_MATRIX}
MAXIT = 60000
RTOL = 1e-10


def listed():
    return [
        # the smallest solve in earnest: a 64 x 64 Poisson problem, where launches
        # and latency count
        {"name": "demo_64", "kind": "demo", "nx": 64, "ny": 64, "mode": "fp64"},
        # the headline problem: 4.2M unknowns in FP64
        {"name": "p1_2048", "kind": "p1", "nx": 2048, "ny": 2048, "mode": "fp64"},
        # the same kind in the FP32-Krylov mode, a ragged rectangle
        {"name": "p1_mixed_1023x770", "kind": "p1", "nx": 1023, "ny": 770, "mode": "mixed"},
        # one eighth of the headline mesh as a strip, FP32 matrix and FP64 vectors
        {"name": "p1_strip_2048x256", "kind": "p1", "nx": 2048, "ny": 256,
         "mode": "mixed_matrix"},
        # a mesh without band structure, as mesh generators give
        {"name": "flipped_300x260", "kind": "flipped", "nx": 300, "ny": 260, "mode": "fp64"},
        # a small cubic problem, odd sizes, element matrices in the reference's order
        {"name": "p3_37x29", "kind": "p3", "nx": 37, "ny": 29, "mode": "fp64", "mfma": False},
        # a large cubic problem, element matrices on the matrix cores
        {"name": "p3_384", "kind": "p3", "nx": 384, "ny": 384, "mode": "fp64", "mfma": True},
        # a parameter study: many uneven linear problems in the mixed mode
        {"name": "batch_p1", "kind": "batch_p1", "nprob": 64, "lo": 32, "hi": 512,
         "mode": "mixed"},
        # many small cubic problems in FP64
        {"name": "batch_p3", "kind": "batch_p3", "nprob": 64, "lo": 8, "hi": 64,
         "mode": "fp64"},
        # one step of a coefficient inversion: two solves and the gradient
        {"name": "adjoint_1024", "kind": "adjoint", "nx": 1024, "ny": 1024, "mode": "fp64"},
        # time stepping: the same two stage matrices, many solves
        {"name": "fkpp_512x384", "kind": "fkpp", "nx": 512, "ny": 384, "steps": 4,
         "mode": "fp64", "nonlocal": False},
        # assembly alone, for a sparse direct solver on the host
        {"name": "handoff_700x500", "kind": "handoff", "nx": 700, "ny": 500},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["demo", "p1", "p1", "p1", "flipped", "p3", "p3", "batch_p1", "batch_p3",
                       "adjoint", "fkpp", "handoff"])
    mode = rng.choice(["fp64", "fp64", "mixed", "mixed_matrix"])
    if kind == "demo":
        return {"kind": kind, "nx": size(8, 200), "ny": size(8, 200), "mode": "fp64"}
    if kind == "p1":
        return {"kind": kind, "nx": size(48, 2048), "ny": size(48, 2048), "mode": mode}
    if kind == "flipped":
        return {"kind": kind, "nx": size(16, 600), "ny": size(16, 600), "mode": mode}
    if kind == "p3":
        return {"kind": kind, "nx": size(8, 384), "ny": size(8, 384), "mode": mode,
                "mfma": rng.random() < 0.5}
    if kind == "batch_p1":
        return {"kind": kind, "nprob": size(3, 64), "lo": size(8, 48), "hi": size(64, 512),
                "mode": mode}
    if kind == "batch_p3":
        return {"kind": kind, "nprob": size(3, 64), "lo": size(4, 12), "hi": size(16, 64),
                "mode": mode}
    if kind == "adjoint":
        return {"kind": kind, "nx": size(48, 1024), "ny": size(48, 1024), "mode": mode}
    if kind == "fkpp":
        nonlocal_ = rng.random() < 0.3
        hi = 256 if nonlocal_ else 640
        return {"kind": kind, "nx": size(32, hi), "ny": size(32, hi), "steps": rng.randint(1, 5),
                "mode": "fp64" if nonlocal_ else mode, "nonlocal": nonlocal_}
    return {"kind": kind, "nx": size(16, 1024), "ny": size(16, 1024)}


# ------------------------------------------------------------------ meshes
def rectangle(nx, ny, rng=None, jitter=0.0, flip=False):
    """(xy, cells) of nx x ny squares cut into two counterclockwise triangles;
    x spans [0, 1] and y spans [0, ny / nx] (square mesh cells)."""
    h = 1.0 / nx
    j, i = np.divmod(np.arange((nx + 1) * (ny + 1)), nx + 1)
    xy = np.stack([i * h, j * h], axis=1)
    if jitter:
        inner = (i > 0) & (i < nx) & (j > 0) & (j < ny)
        xy = xy + inner[:, None] * rng.uniform(-jitter * h, jitter * h, xy.shape)
    cj, ci = np.divmod(np.arange(nx * ny, dtype=np.int64), nx)
    a = ci + cj * (nx + 1)
    b, d, e = a + 1, a + nx + 1, a + nx + 2
    cells = np.empty((nx * ny, 2, 3), np.int32)
    cells[:, 0] = np.stack([a, e, d], axis=1)
    cells[:, 1] = np.stack([a, b, e], axis=1)
    if flip:
        f = rng.random(nx * ny) < 0.5
        cells[f, 0] = np.stack([a, b, d], axis=1)[f]
        cells[f, 1] = np.stack([b, e, d], axis=1)[f]
    return xy, cells.reshape(-1, 3)


def on_boundary(nx, ny):
    j, i = np.divmod(np.arange((nx + 1) * (ny + 1)), nx + 1)
    return ((i == 0) | (i == nx) | (j == 0) | (j == ny)).astype(np.uint8)


def boundary_edges(nx, ny):
    """The boundary edges of the rectangle, each from its lower to its higher
    vertex, and whether each lies on the side x = 0."""
    s = nx + 1
    i, j = np.arange(nx), np.arange(ny)
    ev = np.concatenate([np.stack([i, i + 1], 1), np.stack([i + ny * s, i + 1 + ny * s], 1),
                         np.stack([j * s, (j + 1) * s], 1),
                         np.stack([nx + j * s, nx + (j + 1) * s], 1)]).astype(np.int32)
    left = np.concatenate([np.zeros(2 * nx, bool), np.ones(ny, bool), np.zeros(ny, bool)])
    return ev, left


def p3_numbering(nv, cells):
    """(cell_dofs [ncells x 10], ndofs, boundary DOF flags): vertices, two
    DOFs an edge from its lower to its higher vertex, one DOF a cell."""
    nc = cells.shape[0]
    a = cells[:, [0, 1, 2]].astype(np.int64)
    b = cells[:, [1, 2, 0]].astype(np.int64)
    key, inv, cnt = np.unique((np.minimum(a, b) * nv + np.maximum(a, b)).ravel(),
                              return_inverse=True, return_counts=True)
    inv = inv.reshape(nc, 3)
    first = nv + 2 * inv + (a > b)
    second = nv + 2 * inv + (a < b)
    cd = np.empty((nc, 10), np.int64)
    cd[:, :3] = cells
    cd[:, 3:9:2] = first
    cd[:, 4:9:2] = second
    cd[:, 9] = nv + 2 * key.size + np.arange(nc)
    nd = nv + 2 * key.size + nc
    flags = np.zeros(nd, np.uint8)
    e = np.nonzero(cnt == 1)[0]
    flags[key[e] // nv] = flags[key[e] % nv] = 1
    flags[nv + 2 * e] = flags[nv + 2 * e + 1] = 1
    return cd, nd, flags


# ------------------------------------------------------------------ inputs
def inputs(case, seed):
    """The mesh, the boundary flags and the coefficients as host arrays."""
    rng = np.random.default_rng([int(seed), 7])
    k, d = case["kind"], {}
    if k in ("batch_p1", "batch_p3"):
        sizes = np.rint(np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]),
                                           case["nprob"]))).astype(int)
        rng.shuffle(sizes)
        parts, voff, doff = [], 0, [0]
        for n in sizes:
            n = int(n)
            xy, cells = rectangle(n, n, rng, 0.0 if k == "batch_p1" else 0.2)
            if k == "batch_p1":
                cd, nd, fl = cells.astype(np.int64), xy.shape[0], on_boundary(n, n)
            else:
                cd, nd, fl = p3_numbering(xy.shape[0], cells)
            parts.append((xy, cells + voff, cd + doff[-1], fl))
            voff += xy.shape[0]
            doff.append(doff[-1] + nd)
        d["xy"], d["cells"], d["dofs"], d["flags"] = (np.concatenate(p) for p in zip(*parts))
        d["ndofs"], d["offsets"] = doff[-1], np.array(doff, np.int32)
    else:
        nx, ny = case["nx"], case["ny"]
        d["xy"], d["cells"] = rectangle(nx, ny, rng, 0.2 if k in ("flipped", "p3") else 0.0,
                                        k == "flipped")
        if k == "p3":
            d["dofs"], d["ndofs"], d["flags"] = p3_numbering(d["xy"].shape[0], d["cells"])
        else:
            d["dofs"], d["ndofs"] = d["cells"], d["xy"].shape[0]
            d["flags"] = on_boundary(nx, ny)
    ne = d["cells"].shape[0]
    if k == "demo":
        d["a"], d["g"] = rng.uniform(0.5, 2.0), rng.uniform(0.0, 2.0)
        d["f"] = 2.0 * math.pi ** 2 * d["a"] + d["g"]
    elif k == "fkpp":
        d["c"] = 1.2 * rng.uniform(0.8, 1.2, ne)
        d["cap"] = rng.uniform(0.9, 1.1, d["ndofs"])
        at = rng.uniform(0.3, 0.7, 2) * [1.0, case["ny"] / case["nx"]]
        d["u0"] = 0.05 + 0.3 * np.exp(-((d["xy"] - at) ** 2).sum(1) / 0.02)
    else:
        d["theta"] = rng.standard_normal(ne)
        if k in ("p3", "batch_p3"):
            d["f"] = rng.uniform(0.5, 1.5, ne)
        if k == "adjoint":
            d["uobs"] = (1 - d["flags"]) * 0.05 * rng.uniform(0.8, 1.2, d["ndofs"])
        if k == "handoff":
            left = d["xy"][:, 0] == 0.0
            d["flags"] = left.astype(np.uint8)
            ev, on_left = boundary_edges(case["nx"], case["ny"])
            d["edges"], d["robin"] = ev, (~on_left).astype(np.uint8)
            d["eta"] = rng.uniform(0.5, 1.5, ev.shape[0])
            d["h"] = rng.uniform(-1.0, 1.0, ev.shape[0])
    return d


class State:
    """The handles of one program; closed when the program drops them."""

    def __init__(self):
        self.handles = []

    def keep(self, h):
        self.handles.append(h)
        return h

    def vec(self, n_or_array):
        return self.keep(capi.Vec(context(), n_or_array))

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


_CTX = []


def context():
    if not _CTX:
        _CTX.append(capi.Context(0))
    return _CTX[0]


def const(v):
    return capi.coeff(capi.COEFF_CONST, v)


def prepare(case, seed):
    ctx, d, s, k = context(), inputs(case, seed), State(), case["kind"]
    s.case = case
    p3 = k in ("p3", "batch_p3")
    s.mesh = s.keep(capi.Mesh(ctx, d["xy"], d["cells"], *((d["dofs"], d["ndofs"]) if p3 else ())))
    n = s.n = d["ndofs"]
    s.fe = s.keep(capi.FE(ctx, 3 if p3 else 1))
    if k == "fkpp":
        prepare_fkpp(ctx, s, d, case)
        return s
    s.plan = s.keep(capi.Plan(ctx, s.mesh, d["flags"]))
    s.b, s.x = s.vec(n), s.vec(n)
    if k == "demo":
        s.coeffs = (const(d["a"]), const(d["g"]), capi.coeff(capi.COEFF_SINSIN, d["f"]))
        return s
    s.theta = s.vec(d["theta"])
    alpha = capi.coeff(capi.COEFF_EXPCELL, 1.0, s.theta)
    if p3:
        s.f = s.vec(d["f"])
        f = capi.coeff(capi.COEFF_CELL, 1.0, s.f)
    else:
        f = const(1.0) if k in ("batch_p1", "adjoint") else capi.coeff(capi.COEFF_SINSIN, 1.0)
    s.coeffs = (alpha, const(0.0 if k in ("batch_p1", "adjoint") else 1.0), f)
    if k in ("batch_p1", "batch_p3"):
        s.batch = s.keep(capi.Batch(ctx, s.plan.csr, d["offsets"]))
    if k == "adjoint":
        s.mass = s.keep(capi.Plan(ctx, s.mesh, d["flags"]))
        s.mass.assemble(s.fe, const(0.0), const(1.0), None, None)
        s.uobs, s.diff, s.rhs = s.vec(d["uobs"]), s.vec(n), s.vec(n)
        s.lam, s.grad = s.vec(n), s.vec(d["cells"].shape[0])
    if k == "handoff":
        s.edges = s.keep(capi.Edges(ctx, s.mesh, 1, d["edges"]))
        s.plan.set_edges(s.edges, d["robin"], d["robin"])
        s.eta, s.h = s.vec(d["eta"]), s.vec(d["h"])
        s.coeffs += (capi.coeff(capi.COEFF_CELL, 1.0, s.eta), capi.coeff(capi.COEFF_CELL, 1.0, s.h))
    return s


GROWTH, HORIZON = 2.1, 0.05


def prepare_fkpp(ctx, s, d, case):
    from lehrfempp_amd import fisher_kpp
    ev, _ = boundary_edges(case["nx"], case["ny"])
    flags = np.ones(ev.shape[0], np.uint8)
    s.edges = s.keep(capi.Edges(ctx, s.mesh, 1, ev))
    c = s.vec(d["c"])
    h, loss = const(1.0), None
    if case["nonlocal"]:
        h, eta = fisher_kpp.nonlocal_gain(ctx, s.edges, flags)
        loss = fisher_kpp.nonlocal_loss(ctx, s.edges, flags)
        s.keep(eta), s.keep(loss[1])
    A, M = fisher_kpp.assemble_galerkin_matrices(ctx, s.mesh, s.edges, flags,
                                                 capi.coeff(capi.COEFF_CELL, 1.0, c), h, loss)
    s.keep(A), s.keep(M)
    s.stepper = s.keep(fisher_kpp.StrangSplit(ctx, A, M, HORIZON, case["steps"] + 1, GROWTH,
                                              rtol=RTOL, mode=MODES[case["mode"]]))
    s.cap, s.u0 = s.vec(d["cap"]), s.vec(d["u0"])


# ------------------------------------------------------------------ one pass
def solve(s, b, x):
    x.fill(0.0)
    return capi.pcg(context(), s.plan.csr, b, x, rtol=RTOL, mode=MODES[s.case["mode"]],
                    maxit=MAXIT)


def run(s):
    ctx, k = context(), s.case["kind"]
    if k == "fkpp":
        u = s.stepper.Evolution(s.cap, s.u0)
        out = {"u": u.numpy()}
        u.close()
        return out
    if k == "handoff":
        s.plan.assemble_bd(s.fe, *s.coeffs, s.b)
        rp, col, val = s.plan.csr.download()
        return {"row_ptr": rp, "col": col, "val": val, "b": s.b.numpy()}
    if k in ("batch_p1", "batch_p3"):
        s.x.fill(0.0)
        s.batch.assemble_pcg(s.plan, s.fe, *s.coeffs, s.b, s.x, rtol=RTOL, maxit=MAXIT,
                             mode=MODES[s.case["mode"]])
        return {"x": s.x.numpy()}
    s.plan.assemble(s.fe, *s.coeffs, s.b, mfma=s.case.get("mfma", False))
    solve(s, s.b, s.x)
    if k == "adjoint":
        capi.copy(ctx, s.x, s.diff)
        capi.axpby(ctx, -1.0, s.uobs, 1.0, s.diff)
        capi.spmv(ctx, s.mass.csr, s.diff, s.rhs)
        solve(s, s.rhs, s.lam)
        capi.adjoint_gradient(ctx, s.mesh, s.fe, s.theta, s.x, s.lam, s.grad)
        return {"u": s.x.numpy(), "grad": s.grad.numpy()}
    return {"x": s.x.numpy()}


# ------------------------------------------------------------------ sizes
def counts(case):
    """(cells, DOFs, nonzeros, vertices, longest side in cells) to a few percent."""
    k = case["kind"]
    if k in ("batch_p1", "batch_p3"):
        sizes = np.rint(np.exp(np.linspace(math.log(case["lo"]), math.log(case["hi"]),
                                           case["nprob"])))
        sq, nv, side = float((sizes ** 2).sum()), float(((sizes + 1) ** 2).sum()), case["hi"]
    else:
        sq, nv = case["nx"] * case["ny"], (case["nx"] + 1) * (case["ny"] + 1)
        side = max(case["nx"], case["ny"])
    if k in ("p3", "batch_p3"):
        return 2 * sq, 9 * sq, 153 * sq, nv, side
    return 2 * sq, nv, 7 * nv, nv, side


def work(case):
    """Bytes: mesh, coefficient and element DOFs read once, matrix and load
    vector written once and read once by the solve, the solution written once.
    Operations: the element matrices and, for each iteration (about 4.5 per
    mesh cell along the longest side for P1 and 25 for P3, fewer in one time
    step), a product and five vector updates."""
    ne, n, nnz, nv, side = counts(case)
    k = case["kind"]
    p3 = k in ("p3", "batch_p3")
    nloc = 10 if p3 else 3
    mesh = 16 * nv + (12 + (4 * nloc if p3 else 0) + 8) * ne
    matrix = 12 * nnz + 4 * n
    element = ne * (10 * nloc * nloc + 60)
    iteration = 2 * nnz + 10 * n
    iters = (25 if p3 else 4.5) * side
    if k == "handoff":
        return {"bytes": mesh + matrix + 8 * n, "flops": element}
    if k == "fkpp":
        solves = 2 * max(1, case["steps"])
        return {"bytes": 2 * matrix + 24 * n, "flops": solves * 0.25 * iters * iteration}
    solves = 2 if k == "adjoint" else 1
    if k in ("batch_p1", "batch_p3"):
        iters *= 0.5
    return {"bytes": mesh + 2 * matrix + 24 * n + (8 * ne + 16 * n if solves == 2 else 0),
            "flops": element + solves * iters * iteration}


# ------------------------------------------------------------------ 64 bits
# The same results from plain torch in FP64 (on the GPU where there is one):
# element matrices by the textbook formulas, a coordinate-format sum, and
# conjugate gradients to a residual four orders below the cases' own.
def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def t64(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=device())


def p3_reference():
    """Values and gradients of the cubic shape functions at the points of a
    5 x 5 rule on the unit triangle that integrates degree 6 exactly."""
    g, w = np.polynomial.legendre.leggauss(5)
    g, w = 0.5 * (g + 1), 0.5 * w
    X = np.repeat(g, 5)
    Y = np.tile(g, 5) * (1 - X)
    W = np.repeat(w, 5) * np.tile(w, 5) * (1 - X)
    v = np.array([[0, 0], [1, 0], [0, 1]], float)
    nodes = [v[0], v[1], v[2]]
    for a, b in ((0, 1), (1, 2), (2, 0)):
        nodes += [v[a] + (v[b] - v[a]) / 3, v[a] + 2 * (v[b] - v[a]) / 3]
    nodes = np.array(nodes + [np.array([1 / 3, 1 / 3])])
    pw = [(p, q) for p in range(4) for q in range(4 - p)]
    mono = lambda x, y: np.stack([x ** p * y ** q for p, q in pw], -1)  # noqa: E731
    C = np.linalg.inv(mono(nodes[:, 0], nodes[:, 1]))
    dx = np.stack([p * X ** max(p - 1, 0) * Y ** q for p, q in pw], -1) @ C
    dy = np.stack([q * X ** p * Y ** max(q - 1, 0) for p, q in pw], -1) @ C
    return W, mono(X, Y) @ C, dx, dy


def element_terms(d, alpha, gamma):
    """Element matrices [ne, nloc, nloc] for alpha per cell and constant gamma."""
    V = t64(d["xy"])[torch.as_tensor(d["cells"].astype(np.int64), device=device())]
    e1, e2 = V[:, 1] - V[:, 0], V[:, 2] - V[:, 0]
    det = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0]
    gx = torch.stack([e2[:, 1], -e2[:, 0]], 1) / det[:, None]
    gy = torch.stack([-e1[:, 1], e1[:, 0]], 1) / det[:, None]
    b00, b11, b01 = (gx * gx).sum(1), (gy * gy).sum(1), (gx * gy).sum(1)
    if d["dofs"].shape[1] == 3:
        dx, dy = np.array([[-1.0, 1.0, 0.0]]), np.array([[-1.0, 0.0, 1.0]])
        W, mass = np.array([0.5]), (np.ones((3, 3)) + np.eye(3)) / 24
    else:
        W, N, dx, dy = p3_reference()
        mass = np.einsum("k,ki,kj->ij", W, N, N)
    Kxx, Kyy, Kxy = (np.einsum("k,ki,kj->ij", W, p, q) for p, q in ((dx, dx), (dy, dy), (dx, dy)))
    c = det.abs()
    out = (alpha * c * b00)[:, None, None] * t64(Kxx)
    out += (alpha * c * b11)[:, None, None] * t64(Kyy)
    out += (alpha * c * b01)[:, None, None] * t64(Kxy + Kxy.T)
    if gamma:
        out += (gamma * c)[:, None, None] * t64(mass)
    return out, V, c


def load_p1(V, c, f):
    """Element loads by the three-point rule of degree 2."""
    out = torch.zeros(V.shape[0], 3, dtype=torch.float64, device=V.device)
    for k in range(3):
        lam = [1 / 6] * 3
        lam[k] = 2 / 3
        p = lam[0] * V[:, 0] + lam[1] * V[:, 1] + lam[2] * V[:, 2]
        w = c * f(p) / 6
        for i in range(3):
            out[:, i] += lam[i] * w
    return out


def sinsin(value):
    return lambda p: value * torch.sin(math.pi * p[:, 0]) * torch.sin(math.pi * p[:, 1])


def edge_terms(d, ev, eta, h):
    """Edge mass matrices and loads for coefficients constant on each edge."""
    e = t64(d["xy"])[torch.as_tensor(ev.astype(np.int64), device=device())]
    length = (e[:, 1] - e[:, 0]).norm(dim=1)
    mass = (t64(eta) * length / 6)[:, None, None] * t64([[2.0, 1.0], [1.0, 2.0]])
    load = (t64(h) * length / 2)[:, None].expand(-1, 2)
    return mass, load


def summed(n, parts, fixed):
    """(row_ptr, col, val) of the sum of (dofs, element matrices), rows and
    columns of the fixed DOFs replaced by a unit diagonal."""
    keys, vals = [], []
    for dofs, mats in parts:
        dofs = torch.as_tensor(dofs.astype(np.int64), device=device())
        keys.append((dofs[:, :, None] * n + dofs[:, None, :]).reshape(-1))
        vals.append(mats.reshape(-1))
    key, val = torch.cat(keys), torch.cat(vals)
    free = torch.as_tensor(fixed == 0, device=device())
    keep = free[key // n] & free[key % n]
    at = torch.nonzero(~free).reshape(-1)
    key = torch.cat([key[keep], at * (n + 1)])
    val = torch.cat([val[keep], torch.ones_like(at, dtype=torch.float64)])
    key, inv = torch.unique(key, return_inverse=True)
    val = torch.zeros(key.numel(), dtype=torch.float64, device=key.device).index_add_(0, inv, val)
    rp = torch.searchsorted(key // n, torch.arange(n + 1, device=key.device))
    return rp, key % n, val


def scatter(n, parts, fixed):
    b = torch.zeros(n, dtype=torch.float64, device=device())
    for dofs, vecs in parts:
        b.index_add_(0, torch.as_tensor(dofs.astype(np.int64), device=device()).reshape(-1),
                     vecs.reshape(-1))
    b[torch.as_tensor(fixed != 0, device=device())] = 0.0
    return b


class Matrix:
    """A CSR matrix padded to rows of equal length, with a dense block on some
    rows and columns beside it."""

    def __init__(self, n, csr, block=None):
        rp, col, val = csr
        self.block = block
        rows = torch.repeat_interleave(torch.arange(n, device=rp.device), rp.diff())
        at = torch.arange(col.numel(), device=rp.device) - rp[rows]
        width = int(rp.diff().max())
        self.col = torch.zeros(width, n, dtype=torch.int64, device=rp.device)
        self.val = torch.zeros(width, n, dtype=torch.float64, device=rp.device)
        self.col[at, rows], self.val[at, rows] = col, val
        self.diag = torch.zeros(n, dtype=torch.float64, device=rp.device)
        on = rows == col
        self.diag[rows[on]] = val[on]
        if block is not None:
            self.diag[block[0]] += torch.diagonal(block[1])

    def __matmul__(self, x):
        y = (self.val * x[self.col]).sum(0)
        if self.block is not None:
            y[self.block[0]] += self.block[1] @ x[self.block[0]]
        return y

    def solve(self, b, rtol=3e-14):
        x, r = torch.zeros_like(b), b.clone()
        z = r / self.diag
        p, rho, stop = z.clone(), r @ z, float(b.norm()) * rtol
        for it in range(MAXIT):
            q = self @ p
            a = rho / (p @ q)
            x += a * p
            r -= a * q
            if it % 64 == 63 and float(r.norm()) <= stop:
                break
            z = r / self.diag
            new = r @ z
            p = z + (new / rho) * p
            rho = new
        return x


def exact(case, seed):
    d, k = inputs(case, seed), case["kind"]
    n, dofs = d["ndofs"], d["dofs"]
    if k == "fkpp":
        return exact_fkpp(case, d)
    alpha = d["a"] if k == "demo" else torch.exp(t64(d["theta"]))
    gamma = d["g"] if k == "demo" else 0.0 if k in ("batch_p1", "adjoint") else 1.0
    K, V, c = element_terms(d, alpha, gamma)
    if k in ("p3", "batch_p3"):
        W, N, _, _ = p3_reference()
        F = (t64(d["f"]) * c)[:, None] * t64(W @ N)
    elif k in ("batch_p1", "adjoint"):
        F = load_p1(V, c, lambda p: 1.0)
    else:
        F = load_p1(V, c, sinsin(d["f"] if k == "demo" else 1.0))
    mats, loads = [(dofs, K)], [(dofs, F)]
    if k == "handoff":
        on = d["robin"] != 0
        m, l = edge_terms(d, d["edges"][on], d["eta"][on], d["h"][on])
        mats.append((d["edges"][on], m))
        loads.append((d["edges"][on], l))
    csr = summed(n, mats, d["flags"])
    b = scatter(n, loads, d["flags"])
    if k == "handoff":
        return {"row_ptr": None, "col": None, "val": csr[2], "b": b}
    del mats, loads, K, F
    A = Matrix(n, csr)
    x = A.solve(b)
    if k != "adjoint":
        return {"x": x}
    K0, _, c = element_terms(d, 0.0, 1.0)
    M = Matrix(n, summed(n, [(dofs, K0)], d["flags"]))
    lam = A.solve(M @ (x - t64(d["uobs"])))
    S, _, _ = element_terms(d, 1.0, 0.0)
    at = torch.as_tensor(dofs.astype(np.int64), device=device())
    grad = -alpha * (lam[at][:, :, None] * S * x[at][:, None, :]).sum((1, 2))
    return {"u": x, "grad": grad}


def exact_fkpp(case, d):
    n, dofs = d["ndofs"], d["dofs"]
    none = np.zeros(n, np.uint8)
    ev, _ = boundary_edges(case["nx"], case["ny"])
    ne = ev.shape[0]
    K, _, _ = element_terms(d, t64(d["c"]), 0.0)
    Mel, _, _ = element_terms(d, 0.0, 1.0)
    block = None
    if case["nonlocal"]:
        # two Gauss points an edge; g(x, y) = 1 / (1 + |x - y|^2)
        e = t64(d["xy"])[torch.as_tensor(ev.astype(np.int64), device=device())]
        t = t64([0.5 - math.sqrt(3) / 6, 0.5 + math.sqrt(3) / 6])
        pts = e[:, None, 0] + t[None, :, None] * (e[:, None, 1] - e[:, None, 0])
        w = ((e[:, 1] - e[:, 0]).norm(dim=1)[:, None] / 2).expand(-1, 2).reshape(-1)
        pts = pts.reshape(-1, 2)
        G = 1.0 / (1.0 + (pts[:, None, 0] - pts[None, :, 0]) ** 2
                   + (pts[:, None, 1] - pts[None, :, 1]) ** 2)
        phi = torch.stack([1 - t, t], 1)
        eta = (G @ w).reshape(ne, 2)
        mass = torch.zeros(ne, 2, 2, dtype=torch.float64, device=device())
        for q in range(2):
            mass += (w.reshape(ne, 2)[:, q] * eta[:, q])[:, None, None] * torch.outer(phi[q], phi[q])
        rows, at = np.unique(ev.astype(np.int64), return_inverse=True)
        at = torch.as_tensor(at.reshape(ne, 2), device=device())
        P = torch.zeros(2 * ne, rows.size, dtype=torch.float64, device=device())
        for i in range(2):
            P.index_put_((torch.arange(2 * ne, device=device()), at[:, i].repeat_interleave(2)),
                         phi[:, i].repeat(ne) * w, accumulate=True)
        block = (torch.as_tensor(rows, device=device()), P.T.contiguous() @ (G @ P))
    else:
        mass, _ = edge_terms(d, ev, np.ones(ne), np.ones(ne))
    a = summed(n, [(dofs, K), (ev, mass)], none)
    m = summed(n, [(dofs, Mel)], none)
    A = Matrix(n, a, None if block is None else (block[0], -block[1]))
    kappa, tau = 1.0 - 0.5 * math.sqrt(2.0), HORIZON / (case["steps"] + 1)
    cap, u = t64(d["cap"]), t64(d["u0"])
    full = max(case["steps"] + 1 - 2, 0)
    for i in range(full + 1):
        h = 0.5 * tau if i == 0 else tau
        if i < 2:
            S = Matrix(n, (m[0], m[1], m[2] + h * kappa * a[2]),
                       None if block is None else (block[0], -h * kappa * block[1]))
        y = A @ u
        k1 = S.solve(y)
        k2 = S.solve(y - h * (1 - kappa) * (A @ k1))
        u = u - h * (1 - kappa) * k1 - h * kappa * k2
        u = cap / (1 + (cap / u - 1) * math.exp(-GROWTH * (tau if i < full else tau / 2)))
    return {"u": u}
