"""The calls a user of this framework spends time in, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare(case, seed)`` builds what a user's program holds before the call
(bodies on the device, freestream and wake arrays, target points), ``run(state)`` is one pass through the
public entry points, ``work`` the bytes and operations that pass cannot do without, ``tolerance`` how far
another correct FP64 implementation may be, and ``exact`` the same outputs from plain torch in 64 bits.

Kinds and their ranges (``draw`` samples them, sizes over their logarithm):

  analysis   solve + surface velocity + Cp + forces of a small wing: the first look at a design, all latency
  direct     solve with the default FP64 LU, quads and triangles
  mixed      solve with the FP32 LU and FP64 refinement
  krylov     solve with the FP32 Krylov solver and FP64 refinement (large structured lofts)
  gmres      solve with the FP64 GMRES of the reference's solver protocol
  sources    non-lifting source body: solve, then velocity and potential at a survey plane
  polar      one body at many freestreams (fixed wake)
  batch      independent wings of uneven size in one captured batch
  gradient   lift and drag with their gradients with respect to every node and the freestream
  field      velocity of a solved body at off-body points
  duct       watertight ring wing by the least-squares formulation
  surface    post-processing chain of a solved body: U, grad(mu), Cp, forces, loads
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "flowpanel_amd" not in sys.modules:
        pkg = os.path.join(ROOT, "flowpanel.jl_amd")
        spec = importlib.util.spec_from_file_location("flowpanel_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["flowpanel_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["flowpanel_amd"]


# ---------------------------------------------------------------------------- cases
def listed():
    return [
        # a 96-panel wing from solve to forces: what an interactive session or a unit test runs
        {"name": "wing_first_look", "kind": "analysis", "n_chord": 16, "n_span": 6, "tri": False},
        # the 4,800-panel swept wing with the default solver
        {"name": "wing_direct", "kind": "direct", "n_chord": 60, "n_span": 80, "tri": False},
        # the same wing with the mixed-precision LU
        {"name": "wing_mixed", "kind": "mixed", "n_chord": 60, "n_span": 80, "tri": False},
        # the 30,000-panel blended wing body of the benchmark
        {"name": "bwb_krylov", "kind": "krylov", "n_chord": 250, "n_span": 120, "strips": 4, "coarse": 10},
        # a triangulated wing with the FP64 GMRES
        {"name": "wing_gmres", "kind": "gmres", "n_chord": 50, "n_span": 37, "tri": True},
        # sources on a sphere, odd sizes, pole triangles; survey of U and phi on a plane of points
        {"name": "sphere_sources", "kind": "sources", "n_mer": 47, "n_azi": 99, "targets": 2001},
        # angle-of-attack and sideslip sweep of the swept wing
        {"name": "wing_polar", "kind": "polar", "n_chord": 60, "n_span": 80, "freestreams": 64},
        # 16 wings of 1,000 to 12,000 panels, one captured batch
        {"name": "wings_batch", "kind": "batch", "bodies": 16, "least": 1000, "most": 12000},
        # shape gradient of the 10,000-panel optimisation wing
        {"name": "wing_gradient", "kind": "gradient", "n_chord": 100, "n_span": 100},
        # flow-field box around a 10,000-panel blended wing body
        {"name": "bwb_field", "kind": "field", "n_chord": 100, "n_span": 100, "targets": 600001},
        # watertight ring wing, triangles, least squares
        {"name": "duct_lsq", "kind": "duct", "n_contour": 50, "n_theta": 48},
        # surface post-processing of the 10,000-panel blended wing body
        {"name": "bwb_surface", "kind": "surface", "n_chord": 100, "n_span": 100},
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _wing_size(rng, lo, hi, tri=False):
    """n_chord (even, as the section generator asks) x n_span with about lo..hi panels."""
    n = _between(rng, lo, hi) // (2 if tri else 1)
    nc = max(4, 2 * int(round(0.5 * math.sqrt(n * rng.uniform(0.5, 1.6)))))
    return nc, max(2, n // nc)


def draw(rng):
    kind = rng.choice(["analysis", "direct", "mixed", "krylov", "gmres", "sources", "polar", "batch", "gradient", "field",
                       "duct", "surface"])
    c = {"kind": kind}
    if kind in ("analysis", "direct", "mixed", "gmres"):
        lo, hi = {"analysis": (40, 1500), "direct": (200, 8000), "mixed": (200, 11000), "gmres": (400, 6000)}[kind]
        c["tri"] = rng.random() < 0.5
        c["n_chord"], c["n_span"] = _wing_size(rng, lo, hi, c["tri"])
    elif kind == "krylov":
        c["n_chord"] = 10 * rng.randint(4, 25)
        c["n_span"] = max(12, min(120, _between(rng, 1500, 30000) // c["n_chord"]))
        c["strips"] = rng.choice([1, 2, 4])
        c["coarse"] = rng.choice([10, c["n_chord"] // 5, c["n_chord"]])
    elif kind == "sources":
        n = _between(rng, 200, 6000)
        c["n_mer"] = max(4, int(math.sqrt(n * rng.uniform(0.3, 1.0))))
        c["n_azi"] = max(5, n // c["n_mer"])
        c["targets"] = _between(rng, 10, 20000)
    elif kind == "polar":
        c["n_chord"], c["n_span"] = _wing_size(rng, 300, 5000)
        c["freestreams"] = rng.randint(2, 64)
    elif kind == "batch":
        c["bodies"], c["least"], c["most"] = rng.randint(2, 12), rng.randint(300, 1500), rng.randint(2000, 9000)
    elif kind in ("gradient", "surface"):
        c["n_chord"], c["n_span"] = _wing_size(rng, 300, 9000)
    elif kind == "field":
        c["n_chord"], c["n_span"] = _wing_size(rng, 300, 9000)
        c["targets"] = _between(rng, 50, 500000)
    else:
        n = _between(rng, 500, 5000) // 2
        c["n_contour"] = 2 * int(round(0.5 * math.sqrt(n * rng.uniform(0.6, 1.4))))
        c["n_theta"] = max(8, n // c["n_contour"])
    return c


# ---------------------------------------------------------------------------- inputs
def _rng(seed):
    return np.random.Generator(np.random.PCG64(int(seed) % (1 << 32)))


def _section(g):
    return (float(g.uniform(0.0, 0.03)), 0.4, float(g.uniform(0.10, 0.14)))


def _wing(fp, case, g):
    """Swept tapered wing with a cambered section of the seed (the benchmark's planform)."""
    grid, sh = fp.geometry.loft_wing(airfoil=_section(g), n_chord=case["n_chord"], n_span=case["n_span"], span=10.0,
                                     root_chord=1.0, taper=0.5, sweep_deg=float(g.uniform(25.0, 35.0)))
    if case.get("tri"):
        grid, sh = fp.geometry.triangulate(grid, sh)
    return fp.RigidWakeBody(grid, sh)


def _stream(fp, body, V):
    return np.tile(V[:, None], (1, body.ncells)), np.tile(V[:, None], (1, body.nsheddings))


def _solver(fp, case):
    """Solver function and options, as the benchmark and the tests choose them for such a body."""
    kind = case["kind"]
    if kind == "mixed":
        return fp.solve_lu32_ir, {"tol": 1e-10}
    if kind == "krylov":
        return fp.solve_gmres_ir, {"precond_block": case["strips"] * case["n_chord"], "coarse_block": case["coarse"],
                                   "tol": 1e-8, "inner_tol": 1e-6, "restart": 100}
    if kind == "gmres":
        strip = case["n_chord"] * (2 if case["tri"] else 1)
        return fp.solve_gmres, {"memory": 100, "precond_block": min(1024, 4 * strip), "coarse_block": strip}
    if kind == "gradient":
        strips = min(1024, 4 * case["n_chord"])
        return fp.solve_gmres_ir, {"precond_block": strips, "coarse_block": strips, "tol": 1e-12, "inner_tol": 1e-5,
                                   "restart": 100}
    return fp.solve_ludiv, {}


OBJECTIVE = {"probe_offset": 0.02, "probe_length": 1.0, "span_dir": (0, 1, 0), "ref_area": 8.0}


def prepare(case, seed):
    fp, g, kind = _package(), _rng(seed), case["kind"]
    V = fp.direction(float(g.uniform(2.0, 6.0)), float(g.uniform(-2.0, 2.0)))
    s = {"fp": fp, "kind": kind, "V": V}
    s["solver"], s["opts"] = _solver(fp, case)
    if kind == "sources":
        body = fp.NonLiftingBody(fp.geometry.sphere(1.0, case["n_mer"], case["n_azi"]))
        s["U"] = _stream(fp, body, V)[0]
        # a plane of points downstream and around the body
        s["targets"] = np.asfortranarray(np.stack([g.uniform(1.3, 2.5, case["targets"]), g.uniform(-2, 2, case["targets"]),
                                                   g.uniform(-2, 2, case["targets"])]))
    elif kind == "batch":
        bodies, sizes = [], _rng(3)   # the batch's sizes are the case's; sections and sweeps the seed's
        for _ in range(case["bodies"]):
            ar, sweep, n = sizes.uniform(6, 12), g.uniform(0, 35), int(sizes.uniform(case["least"], case["most"]))
            nc = max(10, 2 * int(round(np.sqrt(n / ar))))
            grid, sh = fp.geometry.loft_wing(airfoil=_section(g), n_chord=nc, n_span=max(4, int(round(n / nc))), span=ar * 0.75,
                                             root_chord=1.0, taper=0.5, sweep_deg=sweep)
            b = fp.RigidWakeBody(grid, sh)
            U, D = _stream(fp, b, V)
            fp.solvers.set_freestream(b, U, D, D)
            bodies.append(b)
        s["bodies"], s["batch"] = bodies, fp.BodyBatch(bodies, solver=fp.solve_lu32_ir,
                                                       solver_optargs={"residual_mode": 0, "tol": 1e-10})
        return s
    elif kind == "gradient":
        grid, sh = fp.geometry.loft_wing(airfoil=_section(g), n_chord=case["n_chord"], n_span=case["n_span"], span=8.0,
                                         root_chord=1.0, taper=1.0, sweep_deg=0.0, twist_tip_deg=-3.0)
        body = fp.RigidWakeBody(grid, sh)
    elif kind == "duct":
        c = fp.geometry.naca4(_section(g), case["n_contour"]).T
        d = 1.67
        body = fp.generate_revolution_liftbody(fp.RigidWakeBody, np.c_[c[:, 0] * d * 0.6, c[:, 1] * d * 0.6 + d / 2],
                                               case["n_theta"], formulation=2)
    elif kind in ("krylov", "field", "surface"):
        body = fp.RigidWakeBody(*fp.geometry.bwb(seed=int(seed) % (1 << 32), n_chord=case["n_chord"],
                                                 n_span=case["n_span"]))
    else:
        body = _wing(fp, case, g)
    s["body"] = body
    if kind == "polar":
        k = case["freestreams"]
        al, be = g.uniform(-5, 10, k), g.uniform(-4, 4, k)
        s["U"] = np.repeat(np.stack([fp.direction(a, b) for a, b in zip(al, be)], axis=1)[:, None, :], body.ncells, axis=1)
        s["D"] = _stream(fp, body, np.array([1.0, 0.0, 0.0]))[1]
        s["solver"] = fp.solve_lu32_ir
    elif kind not in ("sources", "gradient"):
        s["U"], s["D"] = _stream(fp, body, V)
    if kind in ("field", "surface"):
        # a solved body: its strengths come from an earlier call of the program
        block = min(1024, 4 * case["n_chord"])
        fp.solve(body, s["U"], s["D"], s["D"], solver=fp.solve_gmres_ir,
                 solver_optargs={"precond_block": block, "coarse_block": case["n_chord"], "tol": 1e-12, "restart": 100})
    if kind == "field":
        X = body.grid.nodes
        lo, hi = X.min(axis=1), X.max(axis=1)
        pad = 0.25 * (hi - lo)
        s["targets"] = np.asfortranarray(g.uniform((lo - pad)[:, None], (hi + pad)[:, None], (3, case["targets"])))
    return s


def run(s):
    fp, kind, body = s["fp"], s["kind"], s.get("body")
    if kind == "batch":
        s["batch"].solve()
        return [b.strength for b in s["bodies"]]
    if kind == "polar":
        return fp.solve_freestreams(body, s["U"], s["D"], s["D"], solver=s["solver"])[0]
    if kind == "gradient":
        r = fp.lift_drag_gradient(body, s["V"], solver=s["solver"], solver_optargs=s["opts"], **OBJECTIVE)
        return {"coefficients": np.array([r["CL"], r["CDi"]]), "dCL_dnodes": r["dCL_dnodes"][0],
                "dCDi_dnodes": r["dCDi_dnodes"][0], "dCL_dUinf": r["dCL_dUinf"], "dCDi_dUinf": r["dCDi_dUinf"]}
    if kind == "field":
        return fp.Uind(body, s["targets"], np.zeros_like(s["targets"]))
    if kind == "sources":
        fp.solve(body, s["U"])
        return [body.strength, fp.Uind(body, s["targets"], np.zeros_like(s["targets"])),
                fp.phi(body, s["targets"], np.zeros(s["targets"].shape[1]))]
    if kind != "surface":
        fp.solve(body, s["U"], s["D"], s["D"], solver=s["solver"], solver_optargs=s["opts"])
        if kind != "analysis":
            return body.strength
    U = fp.calcfield_U(body, body)
    if kind == "analysis":
        return [body.strength, U, fp.calcfield_Cp(body, 1.0), fp.calcfield_F(body, 1.0, 1.225)]
    grad = fp.calcfield_Ugradmu(body)
    fp.addfields(body, "Ugradmu", "U")
    V = s["V"]
    lift = np.cross(V, [0.0, 1.0, 0.0])
    return [U, grad, fp.calcfield_Cp(body, 1.0), fp.calcfield_F(body, 1.0, 1.225),
            fp.calcfield_LDS(body, lift / np.linalg.norm(lift), V)]


# ---------------------------------------------------------------------------- what a pass cannot do without
def _panels(case):
    kind = case["kind"]
    if kind == "sources":
        return case["n_mer"] * case["n_azi"]
    if kind == "duct":
        return 2 * case["n_contour"] * case["n_theta"]
    return case["n_chord"] * case["n_span"] * (2 if case.get("tri") else 1)


def work(case):
    """Floating-point operations of the influences (184 per quad pair, 138 per triangle pair, 195 per source pair)
    and of the dense solve (2/3 n^3 per factorisation, 2 n^2 per Krylov product at the iteration counts such
    bodies need); bytes: nodes, freestreams, targets in, results out."""
    kind = case["kind"]
    if kind == "batch":
        mean, spread = 0.5 * (case["least"] + case["most"]), case["most"] - case["least"]
        n2 = mean ** 2 + spread ** 2 / 12.0
        n3 = mean * (mean ** 2 + spread ** 2 / 4.0)
        return {"bytes": case["bodies"] * 56 * mean, "flops": case["bodies"] * (184 * n2 + 2 / 3 * n3)}
    n = float(_panels(case))
    pair = 138 if case.get("tri") or kind == "duct" else 195 if kind == "sources" else 184
    aic, lu = pair * n * n, 2 / 3 * n ** 3
    io = 56 * n
    if kind == "krylov":
        return {"bytes": io, "flops": aic + 15 * 2 * n * n}
    if kind == "gmres":
        return {"bytes": io, "flops": aic + 25 * 2 * n * n}
    if kind == "polar":
        k = case["freestreams"]
        return {"bytes": 24 * n + 32 * n * k, "flops": aic + lu + 2 * n * n * k}
    if kind == "gradient":
        return {"bytes": 80 * n, "flops": (184 + 180 + 2 * 780) * n * n + 3 * 40 * 2 * n * n}
    if kind == "field":
        return {"bytes": 48 * case["targets"] + 32 * n, "flops": 180 * n * case["targets"]}
    if kind == "sources":
        return {"bytes": io + 56 * case["targets"], "flops": aic + lu + 390 * n * case["targets"]}
    if kind == "surface":
        return {"bytes": io + 104 * n, "flops": 180 * n * n}
    if kind == "analysis":
        return {"bytes": io + 80 * n, "flops": aic + lu + 180 * n * n}
    return {"bytes": io, "flops": aic + lu}


def tolerance(case):
    kind = case["kind"]
    # iterative paths stop at a residual (1e-8, 1.5e-8, 1e-10) times the amplification of the AIC's inverse
    if kind == "krylov":
        return {"rel": 1e-7, "max": 1e-6}
    if kind == "gmres":
        return {"rel": 1e-6, "max": 1e-5}
    if kind in ("mixed", "batch"):
        return {"rel": 1e-8, "max": 1e-7}
    # FP64 results: rounding times the condition of the body (small wings with a sharp trailing edge: 1e-11 seen)
    if kind in ("polar", "gradient", "surface"):
        return {"rel": 5e-10, "max": 2e-8}
    return {"rel": 1e-10, "max": 4e-9}


# ---------------------------------------------------------------------------- the same in plain torch, 64 bits
OFFSET, CUTOFF = 1e-8, 1e-14   # the bodies' kernel offset and cutoff (defaults)
CHUNK = 1 << 22                # target x panel pairs evaluated together


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.array(a), dtype=torch.float64, device=_dev())


class _Panels:
    """Nodes (n x 3, may carry gradients) and cells of equal or mixed vertex count (short cells repeat a vertex)."""

    def __init__(self, body, nodes=None):
        g = body.grid
        nv = np.diff(g.cell_ptr)
        w = int(nv.max())
        pad = np.minimum(np.arange(w)[None, :], nv[:, None] - 1) + g.cell_ptr[:-1, None]
        self.cells = torch.as_tensor(g.cell_idx[pad], device=_dev())
        self.nv = torch.as_tensor(nv, dtype=torch.float64, device=_dev())
        self.width = w
        self.live = torch.arange(w, device=_dev())[None, :] < torch.as_tensor(nv, device=_dev())[:, None]
        self.x = _t(g.nodes.T) if nodes is None else nodes
        self.shed = body.shedding
        self.cell_host = [g.cell_idx[g.cell_ptr[i]:g.cell_ptr[i + 1]] for i in range(g.ncells)] if body.nsheddings else None
        self.offset = body.CPoffset

    def geometry(self):
        """normal, centroid (before the offset), area, in-plane frame (t, o)."""
        p = self.x[self.cells]
        a, b = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
        t = a / a.norm(dim=1, keepdim=True)
        c = torch.linalg.cross(a, b)
        n = c / c.norm(dim=1, keepdim=True)
        o = torch.linalg.cross(n, t)
        live = self.live[:, :, None].to(p.dtype)
        m = (p * live).sum(1) / self.nv[:, None]
        d = ((p - m[:, None]) * live).sum(1) / self.nv[:, None]
        m = m + (d * t).sum(1, keepdim=True) * t + (d * o).sum(1, keepdim=True) * o
        ac = torch.zeros_like(m)
        for k in range(1, self.width - 1):
            ac = ac + torch.linalg.cross(p[:, k] - p[:, 0], p[:, k + 1] - p[:, 0])
        return n, m, 0.5 * ac.norm(dim=1), t, o

    def horseshoes(self):
        """node of pa, node of pb, panel column of every wake horseshoe."""
        rows = []
        for e in range(self.shed.shape[1]):
            pi, na, nb, pj, ma, mb = (int(v) for v in self.shed[:, e])
            rows.append((self.cell_host[pi][na], self.cell_host[pi][nb], pi))
            if pj != -1:
                rows.append((self.cell_host[pj][ma], self.cell_host[pj][mb], pj))
        return [torch.as_tensor(np.array(v, dtype=np.int64), device=_dev()) for v in zip(*rows)]


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _parts(x):
    return x[..., 0], x[..., 1], x[..., 2]


def _safe(mask, v):
    return torch.where(mask, v, torch.ones_like(v))


def _segment(P, a, b):
    """Velocity of unit regularised segments a -> b (component tuples that broadcast) at P."""
    r, q, e = tuple(x - y for x, y in zip(P, a)), tuple(x - y for x, y in zip(P, b)), tuple(y - x for x, y in zip(a, b))
    c = _cross(r, q)
    c2 = _dot(c, c)
    i, j = 1 / (_dot(r, r).sqrt() + OFFSET), 1 / (_dot(q, q).sqrt() + OFFSET)
    proj = _dot(e, tuple(x * i - y * j for x, y in zip(r, q)))
    f = torch.where(c2 > CUTOFF ** 2, proj / (4 * math.pi * (c2 + OFFSET ** 2)), torch.zeros_like(c2))
    return tuple(f * x for x in c)


def _half_line(P, p, d):
    """Velocity of a unit semi-infinite vortex from p along d."""
    s = _dot(tuple(x - y for x, y in zip(P, p)), d)
    foot = tuple(x + s * y for x, y in zip(p, d))
    u = _segment(P, p, foot)
    far = s.abs() > OFFSET
    h = tuple(x - y for x, y in zip(P, foot))
    h2 = _dot(h, h)
    f = torch.where(h2 > CUTOFF ** 2, 1 / (4 * math.pi * (h2 + OFFSET ** 2)), torch.zeros_like(h2))
    return tuple(torch.where(far, x, torch.zeros_like(x)) + f * y for x, y in zip(u, _cross(d, h)))


def _rings(pan, P):
    """Unit-strength ring velocities (tuple of m x N) at P (m x 3)."""
    Pc = tuple(x[:, None] for x in _parts(P))
    v = [_parts(pan.x[pan.cells[:, k]][None]) for k in range(pan.width)]
    u = (0, 0, 0)
    for k in range(pan.width):
        q = _segment(Pc, v[k], v[(k + 1) % pan.width])   # a repeated vertex is a segment of zero length
        u = tuple(x + y for x, y in zip(u, q))
    return u


def _wakes(pan, P, D, shoes):
    Pc = tuple(x[:, None] for x in _parts(P))
    pa, pb = _parts(pan.x[shoes[0]][None]), _parts(pan.x[shoes[1]][None])
    d = tuple(D[c].reshape(1, 1).expand(1, len(shoes[2])) for c in range(3))
    a, s, b = _half_line(Pc, pa, d), _segment(Pc, pa, pb), _half_line(Pc, pb, d)
    return tuple(y - x + z for x, y, z in zip(a, s, b))


def _chunks(m, n):
    step = max(1, CHUNK // max(1, n))
    return [(i, min(m, i + step)) for i in range(0, m, step)]


def _aic(pan, D):
    n, m, _, _, _ = pan.geometry()
    cp = m + pan.offset * n
    shoes = pan.horseshoes() if pan.shed.shape[1] else None
    A = torch.empty((len(cp), len(cp)), dtype=torch.float64, device=_dev())
    for i, j in _chunks(len(cp), len(cp)):
        w = tuple(x[:, None] for x in _parts(n[i:j]))
        A[i:j] = _dot(_rings(pan, cp[i:j]), w)
        if shoes:
            A[i:j].index_add_(1, shoes[2], _dot(_wakes(pan, cp[i:j], D, shoes), w))
    return A, n, cp


def _velocity(pan, P, gamma, D, shoes):
    u = torch.stack([x @ gamma for x in _rings(pan, P)], 1)
    if shoes:
        u = u + torch.stack([x @ gamma[shoes[2]] for x in _wakes(pan, P, D, shoes)], 1)
    return u


def _velocities(pan, P, gamma, D):
    shoes = pan.horseshoes() if pan.shed.shape[1] else None
    return torch.cat([_velocity(pan, P[i:j], gamma, D, shoes) for i, j in _chunks(len(P), len(pan.cells))])


def _kutta(body, cp):
    """Trailing-edge averaging of the body's own pattern, shedding edges in order."""
    out = cp.clone()
    for e in range(body.nsheddings):
        pi, pj = int(body.shedding[0, e]), int(body.shedding[3, e])
        if pj == -1:
            continue
        ids = [pi, pi + 1, pj, pj - 1] if body.kutta == "reference" else [pi, pj]
        mean = sum(out[i] for i in ids) / len(ids)
        out = out.index_put((torch.tensor(ids, device=out.device),), mean.expand(len(ids)))
    return out


def _source_sums(pan, P):
    """Velocity (m x N x 3 as a tuple) and potential of unit constant-source panels at P (Hess and Smith)."""
    n, _, _, t, o = pan.geometry()
    ex, ey, ez = _parts(o), _parts(t), _parts(-n)
    p0 = pan.x[pan.cells[:, 0]]
    dP = tuple(x[:, None] - y[None] for x, y in zip(_parts(P), _parts(p0)))
    loc = [_dot(dP, tuple(c[None] for c in e)) for e in (ex, ey, ez)]
    x, y, z = loc
    v = [tuple(_dot(_parts(pan.x[pan.cells[:, k]] - p0), e)[None] for e in (ex, ey, ez)) for k in range(pan.width)]
    r = [((x - a) ** 2 + (y - b) ** 2 + (z - c) ** 2).sqrt() for a, b, c in v]
    v1 = v2 = v3 = ps = torch.zeros_like(x)
    dtheta = torch.full_like(x, 2 * math.pi)
    on_edge = torch.zeros_like(x)
    for k in range(pan.width):
        q = torch.where(pan.live[:, (k + 1) % pan.width], (k + 1) % pan.width, 0)[None] if k + 1 < pan.width else None
        live = pan.live[:, k][None]
        if q is None:
            b, rq = v[0], r[0]
        else:
            wrap = (q == 0)
            b = tuple(torch.where(wrap, c0, c1) for c0, c1 in zip(v[0], v[k + 1]))
            rq = torch.where(wrap, r[0], r[k + 1])
        a, rk = v[k], r[k]
        d = ((b[0] - a[0]) ** 2 + (b[1] - a[1]) ** 2 + (b[2] - a[2]) ** 2).sqrt()
        dn = torch.where(live, d, torch.ones_like(d))
        S, C = (b[1] - a[1]) / dn, (b[0] - a[0]) / dn
        si, sj = (a[0] - x) * C + (a[1] - y) * S, (b[0] - x) * C + (b[1] - y) * S
        R = (x - a[0]) * S - (y - a[1]) * C
        J = torch.atan2(R * z.abs() * (rk * sj - rq * si), rk * rq * R * R + z * z * sj * si)
        Q = torch.log((rk + rq + d) / (rk + rq - d + OFFSET))
        w = live.to(x.dtype)
        v1, v2, v3 = v1 - w * S * Q, v2 + w * C * Q, v3 - w * J
        ps = ps - w * (R * Q + z.abs() * J)
        dtheta = torch.where(live & ~(R >= 0), torch.zeros_like(dtheta), dtheta)
        on_edge = on_edge + w * (R == 0)
    ps = ps + z.abs() * dtheta
    v3 = (v3 + dtheta) * torch.sign(z) * (on_edge <= 1)
    k4 = 1 / (4 * math.pi)
    u = tuple(k4 * (v1 * a[None] + v2 * b[None] + v3 * c[None]) for a, b, c in zip(ex, ey, ez))
    return u, k4 * ps


def _solve(A, b):
    return torch.linalg.solve(A, b)


def _np(x):
    return x.detach().cpu().numpy()


def _gradient(body, V):
    """CL, CDi and their gradients: the objective by autograd, the solve by its transpose."""
    x = _t(body.grid.nodes.T).requires_grad_(True)
    U = _t(V).requires_grad_(True)
    N = body.ncells

    def direction(u):
        return u / u.norm()

    def probes(pan):
        n, m, area, _, _ = pan.geometry()
        return m + OBJECTIVE["probe_offset"] * OBJECTIVE["probe_length"] * n, n, area

    def coefficients(u, vel, n, area):
        cp = _kutta(body, 1 - (vel ** 2).sum(1) / (u ** 2).sum())
        d = direction(u)
        lift = torch.linalg.cross(d, _t(OBJECTIVE["span_dir"]))
        lift = lift / lift.norm()
        f = -(cp * area)[:, None] * n
        return [(f @ lift).sum() / OBJECTIVE["ref_area"], (f @ d).sum() / OBJECTIVE["ref_area"]]

    with torch.no_grad():
        pan = _Panels(body, x)
        shoes = pan.horseshoes()
        A, n, cp = _aic(pan, direction(U))
        gamma = _solve(A, -(n @ U))
        vel = _velocities(pan, probes(pan)[0], gamma, direction(U)) + U
    v = vel.clone().requires_grad_(True)
    u0 = U.detach().clone().requires_grad_(True)
    _, n0, area0 = probes(_Panels(body, x))
    J = coefficients(u0, v, n0, area0)
    out = []
    gam = gamma.clone().requires_grad_(True)
    for k in range(2):
        gx, gv, gu = torch.autograd.grad(J[k], [x, v, u0], retain_graph=True)
        gu = gu + gv.sum(0)
        gg = torch.zeros_like(gamma)
        for i, j in _chunks(N, N):   # probe velocities
            pan = _Panels(body, x)
            s = (_velocity(pan, probes(pan)[0][i:j], gam, direction(U), shoes) * gv[i:j]).sum()
            a, b, c = torch.autograd.grad(s, [x, gam, U])
            gx, gg, gu = gx + a, gg + b, gu + c
        lam = _solve(A.T.contiguous(), gg)
        for i, j in _chunks(N, N):   # -lambda . (A gamma - b)
            pan = _Panels(body, x)
            nn, m, _, _, _ = pan.geometry()
            w = _velocity(pan, (m + pan.offset * nn)[i:j], gamma, direction(U), shoes) + U
            s = -(lam[i:j, None] * nn[i:j] * w).sum()
            a, c = torch.autograd.grad(s, [x, U])
            gx, gu = gx + a, gu + c
        out.append((float(J[k]), gx, gu))
    return {"coefficients": np.array([out[0][0], out[1][0]]), "dCL_dnodes": _np(out[0][1].T),
            "dCDi_dnodes": _np(out[1][1].T), "dCL_dUinf": _np(out[0][2]), "dCDi_dUinf": _np(out[1][2])}


def exact(case, seed):
    kind = case["kind"]
    if kind == "surface":
        return None   # grad(mu) is defined by the framework's own neighbour walk; U is covered by "analysis" and "field"
    s = prepare(case, seed)
    if kind == "batch":
        D, out = _t(s["V"]), []
        for b in s["bodies"]:
            A, n, _ = _aic(_Panels(b), D)
            out.append(_np(_solve(A, -(n @ D))))
        return out
    body, V = s["body"], _t(s["V"])
    pan = _Panels(body)
    if kind == "gradient":
        return _gradient(body, s["V"])
    if kind == "field":
        return _np(_velocities(pan, _t(s["targets"].T), _t(body.strength), V).T)
    if kind == "sources":
        n, m, _, _, _ = pan.geometry()
        cp = m + pan.offset * n
        A = torch.cat([_dot(_source_sums(pan, cp[i:j])[0], tuple(x[:, None] for x in _parts(n[i:j])))
                       for i, j in _chunks(len(cp), len(cp))])
        sigma = _solve(A, -(n @ V))
        T = _t(s["targets"].T)
        got = [_source_sums(pan, T[i:j]) for i, j in _chunks(len(T), len(cp))]
        return [_np(sigma), _np(torch.cat([torch.stack([x @ sigma for x in u]) for u, _ in got], 1)),
                _np(torch.cat([p @ sigma for _, p in got]))]
    wake = _t([1.0, 0.0, 0.0]) if kind == "polar" else V
    A, n, cp = _aic(pan, wake)
    if kind == "polar":
        return _np(_solve(A, -(n @ _t(s["U"][:, 0, :]))))
    if kind == "duct":
        # the first strength prescribed to zero, the others by least squares
        Q, R = torch.linalg.qr(A[:, 1:])
        g = torch.linalg.solve_triangular(R, (Q.T @ -(n @ V))[:, None], upper=True)[:, 0]
        return _np(torch.cat([torch.zeros_like(g[:1]), g]))
    gamma = _solve(A, -(n @ V))
    if kind != "analysis":
        return _np(gamma)
    U = _velocities(pan, cp, gamma, V) + V
    Cp = _kutta(body, 1 - (U ** 2).sum(1))
    q = 0.5 * 1.225
    F = -(Cp * q * pan.geometry()[2])[:, None] * n
    return [_np(gamma), _np(U.T), _np(Cp), _np(F.T)]
