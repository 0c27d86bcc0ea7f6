"""Workloads of the elasticity assembly and its solvers, each one call sequence of a user's program.

A case is a dict of plain values: ``op`` names the call sequence, ``material``, ``order`` and ``precision``
the assembler, ``nx``, ``ny``, ``nz`` the cells of the Kuhn box mesh (six tets each).  ``listed()`` gives the
standing cases, ``draw(rng)`` further ones of the same ranges; ``prepare`` builds the handle and the inputs,
``run`` is one pass through the public entry points, ``work`` what the pass cannot do without, and ``exact``
the same outputs from plain FP64 torch on the reference formulas (autograd for stress and tangent).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

MATERIAL_SETS = ("NeoHookean", "LinearElasticity", "SaintVenant", "MooneyRivlin")


def listed():
    return [
        # one tiny mesh inside an outer loop (unit cells, design sweeps): launches and latency count
        _case("assemble", "NeoHookean", 1, "fp64", 3, 2, 3, name="assemble_p1_fp64_tiny"),
        # the 20^3 P1 configuration in FP64 through the host-array API, as a CPU solver calls it
        _case("assemble_host", "NeoHookean", 1, "fp64", 20, 20, 20, name="assemble_host_p1_fp64"),
        # the benchmark's P2 NeoHookean assembly, with the launch shape its tuning keeps
        _case("assemble", "NeoHookean", 2, "mixed", 40, 40, 40, gather=128, name="assemble_p2_mixed_large"),
        # linear elasticity in FP64 on an odd-sized mesh, untuned
        _case("assemble", "LinearElasticity", 2, "fp64", 19, 17, 23, name="assemble_p2_le_fp64"),
        # a P1 mesh of about a million tets (transient and cantilever sizes), untuned
        _case("assemble", "NeoHookean", 1, "mixed", 61, 47, 53, name="assemble_p1_mixed_large"),
        # a material outside the factored path
        _case("assemble", "MooneyRivlin", 2, "mixed", 21, 18, 20, name="assemble_p2_mooney_mixed"),
        # the Hessian-vector product a caller's own iterative solver asks for
        _case("hvp", "NeoHookean", 2, "mixed", 33, 35, 31, name="hvp_p2_mixed"),
        # gradient of an objective: static adjoint solve and the material term, host arrays
        _case("adjoint", "NeoHookean", 2, "mixed", 22, 24, 21, name="adjoint_p2_mixed"),
        # implicit Euler forward and its discrete adjoint (Newton-CG inside every step)
        _case("transient", "NeoHookean", 1, "fp64", 14, 13, 15, steps=3, name="transient_p1_fp64"),
        # a line-search evaluation and the derivative terms of an optimisation step at cantilever size
        _case("derivatives", "NeoHookean", 1, "fp64", 80, 40, 40, name="derivatives_p1_fp64"),
        # the projected Hessian of a Newton step from a compressed state, host arrays
        _case("psd", "NeoHookean", 2, "mixed", 14, 13, 15, name="psd_p2_mixed"),
        # many independent static problems of mixed order and material in one handle
        _case("batch", "mixed", 0, "mixed", 9, 9, 9, problems=16, name="batch_mixed"),
    ]


def draw(rng):
    """One more case: sizes log-uniform in each call's range, never a cube of a listed one."""
    op = rng.choice(("assemble", "assemble", "assemble", "assemble_host", "hvp", "derivatives", "adjoint", "psd", "transient", "batch"))
    order = rng.choice((1, 2))
    precision = rng.choice(("mixed", "fp64"))
    material = rng.choice(("NeoHookean", "NeoHookean", "LinearElasticity"))
    most = {"assemble": 500_000, "assemble_host": 60_000, "hvp": 500_000, "derivatives": 700_000, "adjoint": 60_000,
            "psd": 12_000, "transient": 16_000, "batch": 4_000}[op]
    more = {}
    if op in ("assemble", "hvp", "derivatives") and rng.random() < 0.25:
        material, most = rng.choice(MATERIAL_SETS[2:] if op != "derivatives" else ("SaintVenant",)), 50_000
    if op in ("adjoint", "transient"):
        material = "NeoHookean"
    if op == "transient":
        order, precision, more = 1, "fp64", {"steps": rng.randint(2, 3)}
    if op == "psd":
        precision = "mixed"
    if op == "batch":
        order, material, precision, more = 0, "mixed", "mixed", {"problems": rng.randint(5, 20)}
    if order == 2 and op in ("assemble", "hvp", "derivatives"):
        most //= 3
    least = 300 if op in ("assemble", "hvp") else most // 12
    cells = math.exp(rng.uniform(math.log(least / 6), math.log(most / 6)))
    nx = max(1, round(cells ** (1 / 3) * rng.uniform(0.7, 1.4)))
    ny = max(1, round(math.sqrt(cells / nx) * rng.uniform(0.7, 1.4)))
    nz = max(1, round(cells / (nx * ny)))
    return _case(op, material, order, precision, nx, ny, nz, **more)


def _case(op, material, order, precision, nx, ny, nz, **more):
    return {"op": op, "material": material, "order": order, "precision": precision, "nx": nx, "ny": ny, "nz": nz, **more}


# ------------------------------------------------------------------ inputs


@functools.lru_cache(maxsize=32)
def _box(nx, ny, nz, order):
    from polyfem_amd.mesh import kuhn_box
    return kuhn_box(nx, ny, nz, order=order)


def _mesh(case):
    return _box(case["nx"], case["ny"], case["nz"], case["order"])


def _parameters(case, m, seed):
    """Per-element material parameters: Lame pairs of log-normal stiffness, or MooneyRivlin's (c1, c2, k)."""
    from polyfem_amd.mesh import random_lame
    lam, mu = random_lame(m.n_elements, seed=seed)
    if case["material"] == "MooneyRivlin":
        return 0.35 * mu, 0.15 * mu, lam + 2.0 / 3.0 * mu
    return lam, mu


def _state(m, seed, strain=0.05):
    """A displacement with strains of several per cent: a smooth part and nodal noise scaled to the mesh width."""
    rng = np.random.default_rng(seed)
    X = m.nodes
    u = 0.02 * np.sin(2 * np.pi * X[:, [1, 2, 0]] + rng.uniform(0, 2 * np.pi, 3)) * rng.uniform(0.5, 1.0, 3)
    h = 1.0 / (max(m.grid) * m.order)
    return np.ascontiguousarray((u + rng.normal(0.0, strain * h, u.shape)).ravel())


def _assembler(case, m, seed):
    from polyfem_amd import NLAssembler
    par = _parameters(case, m, seed)
    given = {"params": par} if case["material"] == "MooneyRivlin" else {"lame": par}
    a = NLAssembler(case["material"], m, precision=case["precision"], **given)
    if case.get("gather"):
        a.set_tuning("factored", case["gather"], 256)
    a.set_stream(torch.cuda.current_stream().cuda_stream)
    return a


def _clamped(m, pull):
    """Bottom face fixed, top face moved by pull: (fixed dofs, values, the linear ramp that meets them)."""
    from polyfem_amd.mesh import face_nodes
    bot, top = face_nodes(m, 2, 0.0), face_nodes(m, 2, 1.0)
    fixed = np.concatenate([3 * bot[:, None] + np.arange(3), 3 * top[:, None] + np.arange(3)]).ravel()
    values = np.concatenate([np.zeros(3 * bot.size), np.tile([0.0, 0.0, pull], top.size)])
    ramp = np.zeros(m.n_dofs)
    ramp[2::3] = pull * m.nodes[:, 2]
    return fixed, values, ramp


def _inputs(case, seed):
    """Everything that depends on the seed alone, as host arrays."""
    rng = np.random.default_rng(seed + 1)
    op = case["op"]
    if op == "batch":
        return {"problems": _problems(case, seed)}
    m = _mesh(case)
    d = {"mesh": m, "par": _parameters(case, m, seed), "x": _state(m, seed)}
    if op in ("hvp", "derivatives"):
        d["v"] = rng.normal(size=m.n_dofs)
    if op == "adjoint":
        d["fixed"], d["values"], ramp = _clamped(m, 0.05)
        d["x"] = ramp + 0.1 * _state(m, seed)
        d["x"][d["fixed"]] = d["values"]
        d["rhs"] = rng.normal(size=m.n_dofs)
    if op == "psd":
        d["x"][2::3] -= 0.3 * m.nodes[:, 2]
    if op == "transient":
        d["x"] = np.zeros(m.n_dofs)
        phase, size = rng.uniform(0, 2 * np.pi, 3), rng.uniform(0.3, 0.6, 3)
        d["v0"] = np.ascontiguousarray((size * np.sin(2 * np.pi * m.nodes + phase)).ravel())
        d["gx"] = rng.normal(size=m.n_dofs)
        d["gv"] = rng.normal(size=m.n_dofs)
    return d


def _problems(case, seed):
    rng = np.random.default_rng(seed)
    shape = np.random.default_rng(case["nx"] * 10007 + case["ny"] * 101 + case["nz"])  # the meshes belong to the case
    out = []
    for i in range(case["problems"]):
        n = [max(2, round(case[k] * shape.uniform(0.5, 1.5))) for k in ("nx", "ny", "nz")]
        m = _box(*n, 1 + i % 2)
        pull = rng.uniform(0.02, 0.08)
        fixed, values, ramp = _clamped(m, pull)
        E, nu = math.exp(rng.normal(math.log(1e6), 0.5)), rng.uniform(0.3, 0.45)
        lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        out.append({"mesh": m, "material": "LinearElasticity" if (i // 2) % 2 == 0 else "NeoHookean", "lame": (lam, mu),
                    "fixed_dofs": fixed, "fixed_values": values, "x0": ramp})
    return out


def _device(v):
    return torch.from_numpy(v).to("cuda")


def prepare(case, seed):
    from polyfem_amd import BatchSolver, NewtonSolver, NLProblem, TransientSimulation
    d = _inputs(case, seed)
    op = case["op"]
    s = {"op": op}
    if op == "batch":
        s["solver"] = BatchSolver(d["problems"], precision=case["precision"],
                                  newton=NewtonSolver(max_iterations=20, grad_norm=0.0, relative_grad_norm=1e-4,
                                                      cg_max_iterations=2000, cg_tolerance=1e-6))
        return s
    m = d["mesh"]
    a = s["a"] = _assembler(case, m, seed)
    f64 = {"dtype": torch.float64, "device": "cuda"}
    if op in ("assemble", "hvp", "derivatives"):
        s["x"] = _device(d["x"])
        if "v" in d:
            s["v"] = _device(d["v"])
        s["y"] = torch.empty(a.n_dofs, **f64)
        s["e"] = torch.empty((), **f64)
        if op == "assemble":
            s["values"] = torch.empty(a.nnz, dtype=torch.float32 if case["precision"] == "mixed" else torch.float64, device="cuda")
        if op == "derivatives":
            s["material_term"] = torch.empty(2 * m.n_elements, **f64)
            s["shape_term"] = torch.empty(3 * a.n_vertices, **f64)
    else:
        s["x"] = d["x"]
    if op == "adjoint":
        s["rhs"], s["problem"] = d["rhs"], NLProblem(m.n_dofs, d["fixed"], d["values"])
    if op == "transient":
        s["sim"] = TransientSimulation(a, rho=1000.0, dt=1e-3, time_steps=case["steps"], checkpoint_every=2,
                                       newton=NewtonSolver(max_iterations=20, grad_norm=1e-11, cg_max_iterations=5000, cg_tolerance=1e-10))
        s["v0"], s["gx"], s["gv"] = d["v0"], d["gx"], d["gv"]
    return s


def run(s):
    op = s["op"]
    if op == "batch":
        xs, _ = s["solver"].solve()
        return xs
    a = s["a"]
    if op == "assemble":
        a.energy_gradient_hessian_dev(s["x"].data_ptr(), s["e"].data_ptr(), s["y"].data_ptr(), s["values"].data_ptr())
        return {"energy": s["e"], "gradient": s["y"], "hessian": s["values"]}
    if op == "assemble_host":
        e, g, values = a.assemble_energy_gradient_hessian(s["x"])
        return {"energy": e, "gradient": g, "hessian": values}
    if op == "hvp":
        a.hvp_dev(s["x"].data_ptr(), s["v"].data_ptr(), s["y"].data_ptr())
        return {"product": s["y"]}
    if op == "derivatives":
        x, v = s["x"].data_ptr(), s["v"].data_ptr()
        a.energy_dev(x, s["e"].data_ptr())
        a.gradient_dev(x, s["y"].data_ptr())
        a.material_vjp_dev(x, v, s["material_term"].data_ptr())
        a.shape_vjp_dev(x, v, s["shape_term"].data_ptr())
        return {"energy": s["e"], "gradient": s["y"], "material": s["material_term"], "shape": s["shape_term"]}
    if op == "adjoint":
        from polyfem_amd import solve_static_adjoint
        p = solve_static_adjoint(a, s["x"], s["rhs"], s["problem"], max_iterations=2000, tolerance=1e-8)
        return {"adjoint": p, "material": a.force_material_derivative(s["x"], p)}
    if op == "psd":
        return {"hessian": a.hessian_values(s["x"], project_to_psd=True)}
    x_end, v_end = s["sim"].forward(s["x"], s["v0"])
    d_par, d_x0, d_v0 = s["sim"].adjoint(s["gx"], s["gv"], cg_max_iterations=5000, cg_tolerance=1e-12)
    return {"x": x_end, "v": v_end, "d_parameters": d_par, "d_x0": d_x0, "d_v0": d_v0}


# ------------------------------------------------------------------ compulsory work


@functools.lru_cache(maxsize=64)
def _blocks(nx, ny, nz, order):
    """Node pairs that share an element (the 3x3 blocks of the Hessian)."""
    en = _box(nx, ny, nz, order).elem_nodes.astype(np.int64)
    n = int(en.max()) + 1
    pairs = [np.unique(np.minimum(en[:, a], en[:, b]) * n + np.maximum(en[:, a], en[:, b])) for a in range(en.shape[1]) for b in range(a)]
    return n + 2 * np.unique(np.concatenate(pairs)).size


def work(case):
    """Inputs read once and outputs written once; flops of the basis contractions and tangent blocks."""
    op = case["op"]
    if op == "batch":
        # a converged solve applies each problem's operator some hundred times
        works = [_apply_work(p["mesh"], 4) for p in _problems(case, 0)]
        return {"bytes": sum(w["bytes"] for w in works), "flops": sum(100 * w["flops"] for w in works)}
    m = _mesh(case)
    vb = 4 if case["precision"] == "mixed" else 8
    E, nb, nq, n = m.n_elements, m.n_local, m.n_quad, m.n_dofs
    reads = 8 * n + 4 * E * nb + 24 * m.vertices.shape[0] + 2 * vb * E
    if op in ("assemble", "assemble_host", "psd"):
        blocks = _blocks(case["nx"], case["ny"], case["nz"], case["order"])
        outs = 9 * vb * blocks + (8 * n if op != "psd" else 0)
        flops = E * nb * (nb + 1) / 2 * nq * 36.0
        if op == "psd":
            flops += E * 10.0 * (3 * nb) ** 3
        return {"bytes": float(reads + outs), "flops": flops}
    if op == "hvp":
        return _apply_work(m, vb)
    if op == "derivatives":
        return {"bytes": float(reads + 8 * n + 8 * n + 16 * E + 24 * m.vertices.shape[0]), "flops": E * nq * (8.0 * 18 * nb + 900)}
    w = _apply_work(m, vb)
    applications = 300 if op == "adjoint" else 2 * 60 * case["steps"]
    return {"bytes": w["bytes"], "flops": applications * w["flops"]}


def _apply_work(m, vb):
    E, nb, nq, n = m.n_elements, m.n_local, m.n_quad, m.n_dofs
    return {"bytes": float(24 * n + 4 * E * nb + 24 * m.vertices.shape[0] + 2 * vb * E), "flops": E * nq * (3.0 * 18 * nb + 300)}


# ------------------------------------------------------------------ the same in plain FP64 torch


def _reference_rule(order):
    if order == 1:
        return np.full((1, 3), 0.25), np.full(1, 1 / 6)
    a, b = (5 - math.sqrt(5)) / 20, (5 + 3 * math.sqrt(5)) / 20
    return np.array([[a, a, b], [a, b, a], [b, a, a], [a, a, a]]), np.full(4, 1 / 24)


def _reference_gradients(order, pts):
    lam = np.concatenate([1 - pts.sum(1, keepdims=True), pts], axis=1)
    dlam = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    if order == 1:
        return np.repeat(dlam[None], len(pts), 0)
    edges = [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]
    g = [(4 * lam[:, i, None] - 1) * dlam[i] for i in range(4)]
    g += [4 * (lam[:, i, None] * dlam[j] + lam[:, j, None] * dlam[i]) for i, j in edges]
    return np.stack(g, axis=1)


def _energy_density(material, F, p):
    J = torch.linalg.det(F)
    if material == "NeoHookean":
        lam, mu = p
        return mu / 2 * ((F * F).sum((-1, -2)) - 3 - 2 * torch.log(J)) + lam / 2 * torch.log(J) ** 2
    if material == "MooneyRivlin":
        c1, c2, k = p
        C = F.transpose(-1, -2) @ F
        i1 = C.diagonal(dim1=-1, dim2=-2).sum(-1)
        i2 = 0.5 * (i1 ** 2 - (C * C).sum((-1, -2)))
        return c1 * (J ** (-2 / 3) * i1 - 3) + c2 * (J ** (-4 / 3) * i2 - 3) + k / 2 * torch.log(J) ** 2
    lam, mu = p
    H = F - torch.eye(3, dtype=F.dtype, device=F.device)
    strain = 0.5 * (H + H.transpose(-1, -2))
    if material == "SaintVenant":
        strain = strain + 0.5 * H.transpose(-1, -2) @ H
    return lam / 2 * strain.diagonal(dim1=-1, dim2=-2).sum(-1) ** 2 + mu * (strain * strain).sum((-1, -2))


class _Plain:
    """Energy, gradient, tangent products and the derivative terms of one mesh, per (element, point)."""

    def __init__(self, m, material, par):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        f = {"dtype": torch.float64, "device": dev}
        self.m, self.material, self.dev = m, material, dev
        pts, w = _reference_rule(m.order)
        X = torch.from_numpy(m.vertices[m.elem_vertices]).to(**f)
        T = X[:, 1:] - X[:, :1]  # rows: edges from vertex 0
        self.G = torch.einsum("qak,eck->eqac", torch.from_numpy(_reference_gradients(m.order, pts)).to(**f), torch.linalg.inv(T))
        self.Gv = torch.einsum("qak,eck->eqac", torch.from_numpy(_reference_gradients(1, pts)).to(**f), torch.linalg.inv(T))
        self.w = torch.linalg.det(T)[:, None] * torch.from_numpy(w).to(**f)
        self.par = [torch.as_tensor(np.broadcast_to(np.asarray(p, dtype=np.float64), (m.n_elements,)).copy(), device=dev)[:, None] for p in par]
        self.en = torch.from_numpy(m.elem_nodes.astype(np.int64)).to(dev)
        self.eye = torch.eye(3, **f)

    def vector(self, v):
        return torch.as_tensor(v, dtype=torch.float64, device=self.dev)

    def grad_of(self, v):
        return torch.einsum("ead,eqac->eqdc", v.view(-1, 3)[self.en], self.G)

    def to_nodes(self, S):
        loc = torch.einsum("eqdc,eqac,eq->ead", S, self.G, self.w)
        return torch.zeros(self.m.n_nodes, 3, dtype=torch.float64, device=self.dev).index_add_(0, self.en.reshape(-1), loc.reshape(-1, 3)).view(-1)

    def stress(self, F, graph=False, par=None):
        F = F.detach().requires_grad_(True)
        psi = _energy_density(self.material, F, par or self.par)
        return F, psi, torch.autograd.grad(psi.sum(), F, create_graph=graph)[0]

    def energy_gradient(self, x):
        _, psi, P = self.stress(self.eye + self.grad_of(x))
        return (psi.detach() * self.w).sum(), self.to_nodes(P)

    def tangent(self, x):
        """W -> C : W at x."""
        F, _, P = self.stress(self.eye + self.grad_of(x), graph=True)
        return lambda W: torch.autograd.grad(P, F, W, retain_graph=True)[0]

    def element_hessians(self, x):
        m = self.m
        C, nb = self.tangent(x), m.n_local
        H = torch.empty(m.n_elements, 3 * nb, 3 * nb, dtype=torch.float64, device=self.dev)
        for b in range(nb):
            for n in range(3):
                W = torch.zeros_like(self.G[:, :, :3])
                W[:, :, n] = self.G[:, :, b]
                H[:, :, 3 * b + n] = torch.einsum("eqdc,eqac,eq->ead", C(W), self.G, self.w).reshape(m.n_elements, -1)
        return H

    def csc_values(self, H):
        """Sorted CSC values of the assembled element matrices (symmetric pattern)."""
        m, nb = self.m, self.m.n_local
        key = (self.en[:, :, None] * m.n_nodes + self.en[:, None, :]).reshape(-1)
        blocks, slot = torch.unique(key, return_inverse=True)
        row = blocks // m.n_nodes
        deg = torch.bincount(row, minlength=m.n_nodes)
        first = torch.cumsum(deg, 0) - deg
        base, deg3 = (9 * first[row] + 3 * (torch.arange(blocks.numel(), device=self.dev) - first[row]))[slot], 3 * deg[row][slot]
        values = torch.zeros(9 * blocks.numel(), dtype=torch.float64, device=self.dev)
        for r in range(3):
            for c in range(3):
                values.index_add_(0, base + r * deg3 + c, H[:, r::3, c::3].reshape(-1))
        return values

    def material_term(self, x, p):
        F = self.eye + self.grad_of(x)
        zero, one = torch.zeros_like(self.par[0]), torch.ones_like(self.par[0])
        Gp = self.grad_of(p)
        return torch.cat([-((self.stress(F, par=q)[2] * Gp).sum((-1, -2)) * self.w).sum(1) for q in ((one, zero), (zero, one))])

    def shape_term(self, x, p):
        H, Gp = self.grad_of(x), self.grad_of(p)
        P, B = self.stress(self.eye + H)[2], self.tangent(x)(Gp)
        W = H.transpose(-1, -2) @ B + Gp.transpose(-1, -2) @ P - (P * Gp).sum((-1, -2))[..., None, None] * self.eye
        loc = -torch.einsum("eqdc,eqvc,eq->evd", W, self.Gv, self.w)
        ev = torch.from_numpy(self.m.elem_vertices.astype(np.int64)).to(self.dev)
        return torch.zeros(self.m.vertices.shape[0], 3, dtype=torch.float64, device=self.dev).index_add_(0, ev.reshape(-1), loc.reshape(-1, 3)).view(-1)

    def mass(self, rho):
        """v -> M v, the consistent P1 mass: rho |V| (1 + delta_ab) / 20."""
        vol = rho * self.w.sum(1)[:, None, None] / 20

        def apply(v):
            V = v.view(-1, 3)[self.en]
            loc = vol * (V + V.sum(1, keepdim=True))
            return torch.zeros(self.m.n_nodes, 3, dtype=torch.float64, device=self.dev).index_add_(0, self.en.reshape(-1), loc.reshape(-1, 3)).view(-1)
        return apply

    def diagonal(self, x, a=1.0, extra=None):
        """Diagonal of a H + M, for the iterations' preconditioner."""
        d = torch.zeros(self.m.n_nodes * 3, dtype=torch.float64, device=self.dev)
        H = self.element_hessians(x).diagonal(dim1=-1, dim2=-2)
        d.view(-1, 3).index_add_(0, self.en.reshape(-1), H.reshape(-1, 3))
        return a * d if extra is None else a * d + extra

    def solve(self, apply, diag, b, free, tol, most=6000):
        """Jacobi-preconditioned conjugate gradients on the free dofs."""
        y, r = torch.zeros_like(b), b * free
        z = r / diag.abs()
        p, rz, stop = z.clone(), (r * z).sum(), tol * r.norm()
        for k in range(most):
            q = apply(p) * free
            alpha = rz / (p * q).sum()
            y += alpha * p
            r -= alpha * q
            if k % 8 == 7 and bool(r.norm() <= stop):
                break
            z = r / diag.abs()
            rz, old = (r * z).sum(), rz
            p = z + rz / old * p
        return y

    def minimise(self, x, free, tol, weight=1.0, mass=None, target=None, steps=20):
        """Newton on weight E(x) + 1/2 (x - target) M (x - target) over the free dofs."""
        lumped = None if mass is None else mass(torch.ones_like(x))
        g0 = None
        for _ in range(steps):
            g = weight * self.energy_gradient(x)[1] + (mass(x - target) if mass else 0)
            n = float((g * free).norm())
            g0 = g0 or n
            if n <= tol * g0:
                break
            C = self.tangent(x)
            x = x - self.solve(lambda p: weight * self.to_nodes(C(self.grad_of(p))) + (mass(p) if mass else 0),
                               self.diagonal(x, weight, lumped), g, free, 1e-9)
        return x


def exact(case, seed):
    d = _inputs(case, seed)
    op = case["op"]
    if op == "batch":
        return _exact_batch(d["problems"])
    m = d["mesh"]
    r = _Plain(m, case["material"], d["par"])
    x = r.vector(d["x"])
    if op in ("assemble", "assemble_host", "psd"):
        H = r.element_hessians(x)
        if op == "psd":
            w, V = np.linalg.eigh(H.cpu().numpy())
            return {"hessian": r.csc_values(torch.from_numpy((V * np.maximum(w, 0.0)[:, None]) @ V.transpose(0, 2, 1)).to(r.dev))}
        e, g = r.energy_gradient(x)
        return {"energy": float(e) if op == "assemble_host" else e, "gradient": g, "hessian": r.csc_values(H)}
    if op == "hvp":
        return {"product": r.to_nodes(r.tangent(x)(r.grad_of(r.vector(d["v"]))))}
    if op == "derivatives":
        e, g = r.energy_gradient(x)
        v = r.vector(d["v"])
        return {"energy": e, "gradient": g, "material": r.material_term(x, v), "shape": r.shape_term(x, v)}
    free = torch.ones_like(x)
    if op == "adjoint":
        free[torch.from_numpy(d["fixed"]).long().to(r.dev)] = 0
        C = r.tangent(x)
        p = r.solve(lambda q: r.to_nodes(C(r.grad_of(q))), r.diagonal(x), r.vector(d["rhs"]), free, 1e-10)
        return {"adjoint": p, "material": r.material_term(x, p)}
    return _exact_transient(r, case, d, free)


def _exact_transient(r, case, d, free):
    dt, steps, M = 1e-3, case["steps"], r.mass(1000.0)
    x, v = [r.vector(d["x"])], [r.vector(d["v0"])]
    for _ in range(steps):
        target = x[-1] + dt * v[-1]
        x.append(r.minimise(x[-1], free, 1e-12, dt * dt, M, target))
        v.append((x[-1] - x[-2]) / dt)
    gx, gv = r.vector(d["gx"]), r.vector(d["gv"])
    p1, p2 = torch.zeros_like(gx), torch.zeros_like(gx)
    lumped, d_par = M(torch.ones_like(gx)), 0
    for i in range(steps, 0, -1):
        rhs = M(2 * p1 - p2)
        if i == steps:
            rhs = rhs + gx + gv / dt
        if i == steps - 1:
            rhs = rhs - gv / dt
        C = r.tangent(x[i])
        p = r.solve(lambda q: dt * dt * r.to_nodes(C(r.grad_of(q))) + M(q), r.diagonal(x[i], dt * dt, lumped), rhs, free, 1e-13)
        p1, p2 = p, p1
        d_par = d_par + dt * dt * r.material_term(x[i], p)
    return {"x": x[-1], "v": v[-1], "d_parameters": d_par, "d_x0": M(p1 - p2), "d_v0": dt * M(p1)}


def _exact_batch(problems):
    """The converged solutions; problems of one order and material are solved as one mesh of disjoint parts."""
    from types import SimpleNamespace
    out = [None] * len(problems)
    groups = {}
    for i, p in enumerate(problems):
        groups.setdefault((p["mesh"].order, p["material"]), []).append(i)
    for (order, material), members in groups.items():
        nodes, verts, en, ev, lam, mu, x0, free, cut = 0, 0, [], [], [], [], [], [], [0]
        for i in members:
            p, m = problems[i], problems[i]["mesh"]
            en.append(m.elem_nodes + nodes)
            ev.append(m.elem_vertices + verts)
            nodes, verts = nodes + m.n_nodes, verts + m.vertices.shape[0]
            lam.append(np.full(m.n_elements, p["lame"][0]))
            mu.append(np.full(m.n_elements, p["lame"][1]))
            x, f = np.array(p["x0"]), np.ones(m.n_dofs)
            x[p["fixed_dofs"]], f[p["fixed_dofs"]] = p["fixed_values"], 0.0
            x0.append(x)
            free.append(f)
            cut.append(cut[-1] + m.n_dofs)
        whole = SimpleNamespace(order=order, vertices=np.concatenate([problems[i]["mesh"].vertices for i in members]),
                                elem_vertices=np.concatenate(ev), elem_nodes=np.concatenate(en), n_nodes=nodes,
                                n_elements=sum(map(len, en)), n_local=en[0].shape[1])
        r = _Plain(whole, material, (np.concatenate(lam), np.concatenate(mu)))
        x = r.minimise(r.vector(np.concatenate(x0)), r.vector(np.concatenate(free)), 1e-9)
        for k, i in enumerate(members):
            out[i] = x[cut[k]:cut[k + 1]]
    return out
