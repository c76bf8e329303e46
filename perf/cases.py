"""Measured cases of the explicit solver: what a program does with it, through the Python binding of the C-ABI.

Kinds of case:
  "solve"  a solver that is kept: one pass advances it by `steps` explicit steps, as between two outputs of a run, and
           reads back what the output needs: u, v, a, with `energies` the history columns of those steps, with `fields`
           the element fields of the VTK output (through an output snapshot, as the host driver takes them);
  "whole"  a solve from the input arrays to the result: create, run, read u, v, a, release;
  "batch"  independent cubes in one arena, advanced together, then the state of each;
  "serve"  requests submitted to the serving form, then the displacement of each.

Meshes are boxes with moved interior nodes, clamped at z = 0.  The top is pulled: slowly in kept solvers, which start from
a moving state, as a chained solver does; at the benchmark's speed in solves that start from rest and end; by a sudden
displacement that then stays in the batches, which are advanced on and on.  The precision form ("fp32") computes its forces in single precision, and a program
that picks it keeps its results in single precision too.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("v.1.1_amd"))

import mps_gpu as G  # noqa: E402
from mps_gpu import configs  # noqa: E402

RAMP = 100        # steps over which the prescribed top velocity grows to its full value
SCALE = 0.5       # dt over the stable dt
FOREVER = 1 << 40  # step budget of solvers that are kept


def listed():
    solve = dict(kind="solve", elem="hex", prec="fp64", law=0, het=False, energies=0, loads=False, visc=False,
                 fields=False)
    return [
        # the smallest model in use (10^3 cube): a few workgroups, every step waits on launches and latencies
        dict(solve, name="hex 10^3 fp64", nx=10, ny=10, nz=10, steps=200),
        # a component-sized part with odd sides: about 1/20 of the wavefronts the chip can hold
        dict(solve, name="hex 23x17x29 fp64", nx=23, ny=17, nz=29, steps=200),
        # the largest hex model of the benchmark: 1M elements, 8M Gauss points
        dict(solve, name="hex 100^3 fp64", nx=100, ny=100, nz=100, steps=400),
        # a mid-sized model in the precision form
        dict(solve, name="hex 47x41x53 fp32", nx=47, ny=41, nz=53, steps=200, prec="fp32"),
        # energies every step, as *EXTRACTION of DEFO_ENERGY / KIN_ENERGY asks for, with gravity
        dict(solve, name="hex 33x31x35 energies", nx=33, ny=31, nz=35, steps=100, energies=1, loads=True),
        # loads, bulk viscosity and the element fields of a VTK output; per-element materials, Belytschko law
        dict(solve, name="hex 31x27x25 visc loads", nx=31, ny=27, nz=25, steps=100, law=1, het=True, loads=True,
             visc=True, fields=True),
        # the largest tetrahedral model of the benchmark: 3.07M elements with their own materials
        dict(solve, name="tet 80^3x6 fp64", elem="tet", nx=80, ny=80, nz=80, steps=300, het=True),
        # a mid-sized tetrahedral model in the precision form
        dict(solve, name="tet 21x27x25x6 fp32", elem="tet", nx=21, ny=27, nz=25, steps=200, het=True, prec="fp32"),
        # a parameter study: cubes of 6..40 elements a side, stepped together
        dict(kind="batch", name="batch of 20 cubes fp32", prec="fp32", count=20, lo=6, hi=40, steps=128),
        dict(kind="batch", name="batch of 9 cubes fp64", prec="fp64", count=9, lo=6, hi=24, steps=128),
        # a small solve from its input arrays to the result, set-up included
        dict(kind="whole", name="whole solve 11x13x17", nx=11, ny=13, nz=17, steps=500, prec="fp64"),
        # a burst of requests to the serving form
        dict(kind="serve", name="serve 8 requests fp32", prec="fp32", count=8, lo=1000, hi=20000, steps=256),
    ]


def draw(rng):
    def sides(lo, hi):
        ne = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        a, b = rng.uniform(0.6, 1.6), rng.uniform(0.6, 1.6)
        nx = max(3, round((ne * a) ** (1 / 3)))
        ny = max(3, round((ne * b) ** (1 / 3)))
        return nx, ny, max(3, round(ne / (nx * ny)))

    r = rng.random()
    if r < 0.68:
        tet = rng.random() < 0.35
        nx, ny, nz = sides(150, 60000) if tet else sides(300, 300000)
        prec = "fp64" if rng.random() < 0.65 else "fp32"
        law = rng.choice([0, 0, 0, 1, 2, 3])
        extra = rng.random()
        return dict(kind="solve", elem="tet" if tet else "hex", prec=prec, law=law, het=rng.random() < (0.7 if tet else 0.25),
                    energies=rng.choice([1, 5]) if extra < 0.2 else 0, loads=extra < 0.35, visc=0.2 <= extra < 0.35 and not tet,
                    fields=rng.random() < 0.15, nx=nx, ny=ny, nz=nz, steps=rng.randrange(60, 260))
    if r < 0.84:
        prec = "fp64" if rng.random() < 0.5 else "fp32"
        lo = rng.randrange(5, 12)
        return dict(kind="batch", prec=prec, count=rng.randrange(3, 21), lo=lo, hi=lo + rng.randrange(4, 25), steps=32 * rng.randrange(2, 6))
    if r < 0.93:
        nx, ny, nz = sides(300, 20000)
        return dict(kind="whole", nx=nx, ny=ny, nz=nz, steps=rng.randrange(200, 700), prec="fp64" if rng.random() < 0.6 else "fp32")
    return dict(kind="serve", prec="fp32", count=rng.randrange(3, 10), lo=1000, hi=rng.randrange(4000, 20000), steps=32 * rng.randrange(4, 12))


# ---------------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------------
def material(seed, k=0):
    """One material of the benchmark's ranges: E log-uniform in [1e5, 1e7], nu uniform in [0.2, 0.45], rho 1000."""
    u = configs.uniform01(seed ^ configs.MAT_XOR, np.array([2 * k, 2 * k + 1]))
    return float(10.0 ** (5.0 + 2.0 * u[0])), float(0.2 + 0.25 * u[1])


def sound(law, E, nu, rho=1000.0):
    return math.sqrt(E / rho) if law >= 2 else math.sqrt(E * (1 - nu) / ((1 + nu) * (1 - 2 * nu)) / rho)


def box_model(nx, ny, nz, seed, tet=False, law=0, het=False, pull=2e-5):
    """Mesh, material and supports of a box whose longest side is 1: the arrays that a program hands over.  The top moves
    at `pull` times the speed of sound, or (None) is displaced once by 2% of an element."""
    n = max(nx, ny, nz)
    m = configs.perturb(configs.box(nx, ny, nz, nx / n, ny / n, nz / n, tet=tet), 0.15 if tet else 0.10, seed)
    E, nu = configs.random_materials(m["n_elem"], seed, 3e5, 3e6) if het else material(seed)
    c = sound(law, 1e6 if het else E, 0.3 if het else nu)
    dof, val = configs.clamp_bottom_pull_top(m, vel=0.02 / n if pull is None else pull * c)
    return dict(mesh=m, law=law, E=E, nu=nu, rho=1000.0, dir_dof=dof, dir_val=val, c=c,
                bc_mode=G.BC_INST if pull is None else G.BC_VELOCITY)


def moving_state(model, seed):
    """u, v, a of a vibrating body: a few long waves with strains of some 1e-3, zero at the clamped face."""
    m = model["mesh"]
    N = m["n_nodes"]
    x = m["X"].reshape(3, N)
    rng = np.random.default_rng(seed)
    u, v, a = np.zeros((3, N)), np.zeros((3, N)), np.zeros((3, N))
    for _ in range(3):
        k = rng.uniform(1.0, 5.0, 3)
        amp, ph = rng.uniform(-1.0, 1.0, 3), rng.uniform(0.0, 2 * np.pi)
        s = np.sin(k @ x + ph) * x[2]
        for d in range(3):
            u[d] += 1e-3 * amp[d] * s
            v[d] += 2e-3 * model["c"] * amp[(d + 1) % 3] * s
            a[d] -= 2e-3 * model["c"] ** 2 * amp[d] * s
    return u.ravel(), v.ravel(), a.ravel()


def load_list(model):
    """Gravity, a traction on the elements of the top layer's upper faces and a force on the far corner."""
    m = model["mesh"]
    per = m["nx"] * m["ny"]
    p = 1e-4 * 1000.0 * model["c"] ** 2
    out = [("gravity", 9.81)]
    if m["nen"] == 8:
        out.append(("traction_inst", (0.3 * p, -0.2 * p, p), 0.0, 1e9, np.arange(per) + per * (m["nz"] - 1), np.full(per, 2)))
    out.append(("force", [m["n_nodes"] - 1], [[p / per, 0.0, 0.5 * p / per]], 0.0, 10.0))
    return out


def prec_of(case):
    return G.PREC_FP32_ELEM if case["prec"] == "fp32" else G.PREC_FP64


def cubes(case, seed):
    """Sides of the batch's cubes (over the whole range, the same for every seed) and their solves."""
    sides = np.linspace(case["lo"], case["hi"], case["count"]).round().astype(int)
    return [box_model(int(n), int(n), int(n), seed + 977 * k, pull=None) for k, n in enumerate(sides)]


def requests(case, seed):
    """Boxes of lo..hi elements, spread over the logarithm, aspect 1..4 along z, as the serving workload draws them."""
    out = []
    for k in range(case["count"]):
        ne = case["lo"] * (case["hi"] / case["lo"]) ** (k / max(1, case["count"] - 1))
        asp = 1.0 + 3.0 * ((k * 5) % case["count"]) / case["count"]
        nx = max(1, round((ne / asp) ** (1 / 3)))
        out.append(box_model(nx, nx, max(1, round(asp * nx)), seed + 977 * k, pull=2e-3))
    return out


def prepare(case, seed):
    if case["kind"] == "solve":
        md = box_model(case["nx"], case["ny"], case["nz"], seed, case["elem"] == "tet", case["law"], case["het"])
        s = G.Solver(md["mesh"], law=md["law"], E=md["E"], nu=md["nu"], rho=md["rho"], dir_dof=md["dir_dof"],
                     dir_val=md["dir_val"], bc_mode=G.BC_VELOCITY, vel_ramp_steps=RAMP, scale=SCALE, n_steps=FOREVER,
                     precision=prec_of(case), energy_every=case["energies"])
        s.set_state(*moving_state(md, seed))
        if case["loads"]:
            s.set_loads(loads=load_list(md))
        if case["visc"]:
            s.set_viscosity(G.VISC_BULK, c1=0.5, cl=0.06)
        s.prepare_run(case["steps"])
        return dict(case=case, solver=s, done=0)
    if case["kind"] == "whole":
        return dict(case=case, model=box_model(case["nx"], case["ny"], case["nz"], seed, pull=2e-3))
    if case["kind"] == "batch":
        models = cubes(case, seed)
        need = sum(m["mesh"]["n_elem"] + m["mesh"]["n_nodes"] for m in models)
        b = G.Batch(arena_bytes=(64 << 20) + 700 * need, max_instances=len(models), precision=prec_of(case))
        slots = [b.add(m["mesh"], law=m["law"], E=m["E"], nu=m["nu"], rho=m["rho"], dir_dof=m["dir_dof"],
                       dir_val=m["dir_val"], bc_mode=m["bc_mode"], scale=SCALE, n_steps=FOREVER) for m in models]
        b.autotune()
        return dict(case=case, batch=b, slots=slots)
    return dict(case=case, server=G.Server(arena_bytes=1 << 30, max_instances=64, precision=prec_of(case)),
                models=requests(case, seed))


def kept(case, arrays):
    """Results in the precision that the program keeps."""
    return [x.astype(np.float32) for x in arrays] if case["prec"] == "fp32" else list(arrays)


def run(state):
    case = state["case"]
    if case["kind"] == "solve":
        s, first, n = state["solver"], state["done"], case["steps"]
        rc, rep = s.run(n)
        if rc != 0:
            raise RuntimeError(f"solve ended with {rc}: {rep}")
        state["done"] = first + n
        out = {}
        if case["fields"]:
            s.snapshot_begin(0, True)
            u, v, a, el = s.snapshot_wait(0)
            s.snapshot_release(0)
            out["fields"] = el
        else:
            u, v, a = s.get_state()
        out["state"] = kept(case, (u, v, a))
        out["time"], out["dt"] = (np.array([rep["time"]]), np.array([rep["dt"]])) if case["prec"] == "fp64" else \
            (np.float32([rep["time"]]), np.float32([rep["dt"]]))
        if case["fields"] and case["prec"] == "fp32":
            out["fields"] = out["fields"].astype(np.float32)
        if case["energies"]:
            h = s.history(first, n)
            h.update(s.energy_balance(first, n))
            keys = ("e_def", "e_kin", "volume", "e_ext", "e_kin_lumped", "w_ext", "w_react")
            out["history"] = kept(case, [h[k] for k in keys])
        return out
    if case["kind"] == "whole":
        m = state["model"]
        with G.Solver(m["mesh"], law=m["law"], E=m["E"], nu=m["nu"], rho=m["rho"], dir_dof=m["dir_dof"],
                      dir_val=m["dir_val"], vel_ramp_steps=RAMP, scale=SCALE, n_steps=case["steps"],
                      precision=prec_of(case)) as s:
            rc, rep = s.run(case["steps"])
            if rc != 0:
                raise RuntimeError(f"solve ended with {rc}: {rep}")
            return kept(case, s.get_state())
    if case["kind"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        return [kept(case, b.get_state(k)) for k in state["slots"]]
    srv = state["server"]
    ids = [srv.submit(m["mesh"], law=m["law"], E=m["E"], nu=m["nu"], rho=m["rho"], dir_dof=m["dir_dof"],
                      dir_val=m["dir_val"], vel_ramp_steps=RAMP, scale=SCALE, n_steps=case["steps"])
           for m in state["models"]]
    out = []
    for i in ids:
        rc, u, _, _ = srv.result(i)
        if rc != 0:
            raise RuntimeError(f"request {i} ended with {rc}")
        out.append(u)
    return kept(case, out)


# ---------------------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def step_work(nx, ny, nz, tet, prec, het, energies=0, visc=False):
    """One explicit step: every step reads the mesh (connectivity, X, undeformed length, materials, lumped mass) and the
    state u, v once and writes u, v once; the result's last acceleration is small beside that.  Operations of a Gauss
    point: J and grad u (2 x 72 by sum factorisation), cofactors, determinant, H, the law, the stress in the reference
    frame and its moments, about 330; of an element the transforms, about 250."""
    ne, nn = nx * ny * nz * (6 if tet else 1), (nx + 1) * (ny + 1) * (nz + 1)
    nen = 4 if tet else 8
    b = ne * (4 * nen + 8 + (24 if het else 0)) + nn * (24 + 8 + 4 * 24)
    f = ne * (330 + 150 if tet else 8 * 330 + 250) + nn * 20
    if visc:
        b, f = b + 24 * nn, f + ne * 8 * 60
    if energies:
        b, f = b + 24 * nn / energies, f + ne * (60 if tet else 8 * 70) / energies
    return b, f


def work(case):
    k = case["kind"]
    p = case["prec"]
    if k in ("solve", "whole"):
        tet, het = case.get("elem") == "tet", case.get("het", False)
        b, f = step_work(case["nx"], case["ny"], case["nz"], tet, p, het, case.get("energies", 0), case.get("visc", False))
        nn = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
        out = 9 * nn * 8 + (case["nx"] * case["ny"] * case["nz"] * (6 if tet else 1) * 168 if case.get("fields") else 0)
        return {"bytes": case["steps"] * b + out, "flops": case["steps"] * f}
    if k == "batch":
        sides = np.linspace(case["lo"], case["hi"], case["count"]).round().astype(int)
        w = [step_work(n, n, n, False, p, False) for n in map(int, sides)]
        out = sum(72 * (n + 1) ** 3 for n in map(int, sides))
    else:
        ms = requests(case, 1)
        w = [step_work(m["mesh"]["nx"], m["mesh"]["ny"], m["mesh"]["nz"], False, p, False) for m in ms]
        out = sum(24 * m["mesh"]["n_nodes"] for m in ms)
    return {"bytes": float(case["steps"] * sum(b for b, _ in w) + out), "flops": float(case["steps"] * sum(f for _, f in w))}


# ---------------------------------------------------------------------------------------------------------------------
# The same in plain 64-bit torch
# ---------------------------------------------------------------------------------------------------------------------
class Plain:
    """The explicit solve with torch in float64: isoparametric hex8 (2x2x2 Gauss) and tet4 elements, row-sum lumped
    mass, central differences, the stable step from the deformed inscribed-sphere length."""

    def __init__(self, model, loads=None, visc=False):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        m = model["mesh"]
        self.dev, self.N, self.law = dev, m["n_nodes"], model["law"]
        self.nen = nen = m["nen"]
        t = lambda x, dt=torch.float64: torch.as_tensor(np.asarray(x), dtype=dt, device=dev)  # noqa: E731
        self.X = t(m["X"]).reshape(3, -1)
        self.conn = t(m["conn"], torch.int64).reshape(-1, nen).t().contiguous()  # [nen, E]
        E, nu = t(np.broadcast_to(model["E"], (m["n_elem"],)).copy()), t(np.broadcast_to(model["nu"], (m["n_elem"],)).copy())
        self.rho = model["rho"]
        self.lam, self.mu, self.K = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu)), E / (3 * (1 - 2 * nu))
        self.c = torch.sqrt((E if self.law >= 2 else self.lam + 2 * self.mu) / self.rho)
        # shape values and natural derivatives at the Gauss points, with the rule's own literals
        if nen == 8:
            g = 0.577350269
            sg = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], float)
            phi = np.prod(1 + sg[None] * (g * sg)[:, None], axis=2) / 8
            nd = np.empty((8, 8, 3))
            for j in range(3):
                o = [i for i in range(3) if i != j]
                nd[:, :, j] = sg[None, :, j] * np.prod(1 + sg[None][:, :, o] * (g * sg)[:, None][:, :, o], axis=2) / 8
            w = 1.0
        else:
            phi = np.full((1, 4), 0.25)
            nd = np.array([[[-1, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]]], float)
            w = 0.166666666667
        self.phi, nd = t(phi), t(nd)
        x = self.X[:, self.conn]  # [3, nen, E]
        self.D, self.wJ = [], []
        mass = torch.zeros(nen, m["n_elem"], dtype=torch.float64, device=dev)
        for q in range(nd.shape[0]):
            J = [[(x[i] * nd[q, :, j].unsqueeze(1)).sum(0) for j in range(3)] for i in range(3)]
            C, det = self.cof(J)
            self.D.append(torch.stack([sum(nd[q, :, k].unsqueeze(1) * (C[j][k] / det) for k in range(3)) for j in range(3)]))
            self.wJ.append(w * det.abs())
            mass += self.wJ[q] * self.rho * self.phi[q].unsqueeze(1)  # sum_b phi_b = 1
        self.mass = self.scatter(mass)
        self.l0 = self.length(x)
        self.visc = visc
        self.fixed, self.val, self.inst = t(model["dir_dof"], torch.int64), t(model["dir_val"]), model["bc_mode"] == G.BC_INST
        self.fext_at = self.external(model, loads or [])
        self.u, self.v, self.a = (torch.zeros(3, self.N, dtype=torch.float64, device=dev) for _ in range(3))
        self.k, self.time, self.dt = 0, 0.0, SCALE * float((self.l0 / self.c).min())
        self.rows, self.we, self.wr, self.fp, self.rp = [], 0.0, 0.0, None, None

    @staticmethod
    def cof(A):
        C = [[A[(i + 1) % 3][(j + 1) % 3] * A[(i + 2) % 3][(j + 2) % 3] - A[(i + 1) % 3][(j + 2) % 3] * A[(i + 2) % 3][(j + 1) % 3]
              for j in range(3)] for i in range(3)]
        return C, A[0][0] * C[0][0] + A[0][1] * C[0][1] + A[0][2] * C[0][2]

    def scatter(self, f):
        """Sum of element-node values f[nen, E] at the nodes."""
        out = torch.zeros(self.N, dtype=torch.float64, device=self.dev)
        return out.index_add_(0, self.conn.reshape(-1), f.reshape(-1))

    def length(self, x):
        """Twice the inscribed-sphere radius 3V/A: the sum of the face triangles, the volume of the corner's edges."""
        def cross(a, b):
            return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])
        P = [x[:, k] for k in range(self.nen)]
        if self.nen == 8:
            quads = [(0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (0, 3, 7, 4)]
            tris = [t for q in quads for t in ((q[0], q[1], q[2]), (q[0], q[2], q[3]))]
            c, f = (1, 3, 4), 1.0
        else:
            tris, c, f = [(0, 1, 2), (1, 2, 3), (0, 2, 3), (0, 1, 3)], (1, 2, 3), 1.0 / 6.0
        A = sum(0.5 * cross(P[p] - P[r], P[q] - P[r]).square().sum(0).sqrt() for p, q, r in tris)
        V = f * ((P[c[0]] - P[0]) * cross(P[c[1]] - P[0], P[c[2]] - P[0])).sum(0).abs()
        return 6.0 * V / A

    def external(self, model, loads):
        """External force as a function of time: gravity, dead tractions on hex faces 2, nodal forces."""
        base = torch.zeros(3, self.N, dtype=torch.float64, device=self.dev)
        nodal = []
        for b in loads:
            if b[0] == "gravity":
                base[2] += self.scatter(sum(-self.wJ[q] * self.rho * b[1] * self.phi[q].unsqueeze(1) for q in range(len(self.wJ))))
            elif b[0] == "force":
                nodal.append((b[1][0], torch.as_tensor(b[2][0], dtype=torch.float64, device=self.dev) / (b[4] - b[3])))
            else:  # traction on the flat face 4, 7, 6, 5: w |J_s| phi_a T
                el = torch.as_tensor(b[4], device=self.dev)
                nodes = self.conn[:, el][[4, 7, 6, 5]].t()
                x = self.X[:, nodes]
                g = 0.577350269
                s4 = np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], float)
                for p in s4 * g:
                    ph = torch.as_tensor((1 + s4[:, 0] * p[0]) * (1 + s4[:, 1] * p[1]) / 4, device=self.dev)
                    d0 = torch.as_tensor(s4[:, 0] * (1 + s4[:, 1] * p[1]) / 4, device=self.dev)
                    d1 = torch.as_tensor(s4[:, 1] * (1 + s4[:, 0] * p[0]) / 4, device=self.dev)
                    a0, a1 = (x * d0).sum(2), (x * d1).sum(2)
                    Js = torch.linalg.cross(a0.t(), a1.t()).norm(dim=1)
                    for i in range(3):
                        base[i].index_add_(0, nodes.reshape(-1), (Js.unsqueeze(1) * ph * b[1][i]).reshape(-1))

        def at(time):
            f = base
            if nodal:
                f = base.clone()
                for n, rate in nodal:
                    f[:, n] += rate * time
            return f
        return at

    def stress(self, H):
        """First Piola-Kirchhoff stress, energy density and det F of a law from H = F - I."""
        d = lambda i, j: 1.0 if i == j else 0.0  # noqa: E731
        F = [[H[i][j] + d(i, j) for j in range(3)] for i in range(3)]
        C, J = self.cof(F)
        R = range(3)
        if self.law == 0:
            l = torch.log(J)
            s = (self.lam * l - self.mu) / J
            W = 0.5 * self.lam * l * l - self.mu * l + 0.5 * self.mu * sum(F[i][j] * F[i][j] for i in R for j in R)
            return F, C, J, [[self.mu * F[i][j] + s * C[i][j] for j in R] for i in R], W
        if self.law == 1:
            B = [[sum(F[i][k] * F[j][k] for k in R) for j in R] for i in R]
            r = J ** (-5.0 / 3.0)
            p = -(self.mu / 3) * (B[0][0] + B[1][1] + B[2][2]) * r + self.K * (J - 1)
            S = [[self.mu * r * B[i][j] + (p if i == j else 0.0) for j in R] for i in R]
            return F, C, J, [[sum(S[i][k] * C[k][j] for k in R) for j in R] for i in R], torch.zeros_like(J)
        E = [[0.5 * (H[i][j] + H[j][i] + (sum(H[k][i] * H[k][j] for k in R) if self.law == 2 else 0.0)) for j in R] for i in R]
        tr = self.lam * (E[0][0] + E[1][1] + E[2][2])
        S = [[2 * self.mu * E[i][j] + (tr if i == j else 0.0) for j in R] for i in R]
        W = 0.5 * sum(S[i][j] * E[i][j] for i in R for j in R)
        if self.law == 3:
            return F, C, J, S, W
        return F, C, J, [[sum(F[i][k] * S[k][j] for k in R) for j in R] for i in R], W

    def grad(self, x, q):
        return [[(x[i] * self.D[q][j]).sum(0) for j in range(3)] for i in range(3)]

    def forces(self, u, du=None, dt=0.0):
        """Internal force; the step's deformation energy and volume."""
        x = u[:, self.conn]
        f = [torch.zeros(self.nen, self.conn.shape[1], dtype=torch.float64, device=self.dev) for _ in range(3)]
        ed, vol = 0.0, 0.0
        for q in range(len(self.wJ)):
            F, C, J, P, W = self.stress(self.grad(x, q))
            if self.visc:
                d = self.grad(du[:, self.conn], q)
                tr = (d[0][0] + d[1][1] + d[2][2]) / dt
                z = self.rho / J * self.l0 * (0.25 * self.l0 * tr.abs() * tr.clamp(max=0.0) + 0.06 * self.c * tr)
                P = [[P[i][j] + z * C[i][j] for j in range(3)] for i in range(3)]
            for i in range(3):
                f[i] += self.wJ[q] * (P[i][0] * self.D[q][0] + P[i][1] * self.D[q][1] + P[i][2] * self.D[q][2])
            ed, vol = ed + (self.wJ[q] * W).sum(), vol + (self.wJ[q] * J).sum()
        return torch.stack([self.scatter(y) for y in f]), ed, vol

    def step(self, energies=False):
        k = self.k = self.k + 1
        self.time += self.dt
        dt = self.dt = SCALE * float((torch.minimum(self.l0, self.length((self.X + self.u)[:, self.conn])) / self.c).min())
        du = dt * self.v + 0.5 * dt * dt * self.a
        if self.inst:  # displaced once, at the first step
            V = U = self.val * (1.0 if k == 1 else 0.0)
        else:
            V = self.val * min(k / RAMP, 1.0)
            U = V * dt
        du.view(-1)[self.fixed] = U
        vold = self.v.view(-1)[self.fixed].clone()
        self.u = self.u + du
        fi, ed, vol = self.forces(self.u, du, dt)
        fe = self.fext_at(self.time)
        a = (fe - fi) / self.mass
        a.view(-1)[self.fixed] = 0.0
        self.v = self.v + 0.5 * dt * (self.a + a)
        self.v.view(-1)[self.fixed] = V
        self.a = a
        if energies:
            r = (fi - fe).reshape(-1)[self.fixed]
            m = self.mass.repeat(3)[self.fixed]
            if k >= 2:
                self.we += float((0.5 * (self.fp + fe) * du).sum())
                self.wr += float((0.5 * (self.rp + r) * du.view(-1)[self.fixed] + 0.5 * m * (V * V - vold * vold)).sum())
            self.fp, self.rp = fe, r
            ek = 0.0
            vn = self.v[:, self.conn]
            for q in range(len(self.wJ)):
                vq = (vn * self.phi[q].unsqueeze(1)).sum(1)
                ek += (0.5 * self.rho * self.wJ[q] * vq.square().sum(0)).sum()
            self.rows.append([float(ed), float(ek), float(vol), float((self.u * fe).sum()),
                              float(0.5 * (self.mass * self.v.square()).sum()), self.we, self.wr])

    def fields(self):
        """Gauss-point averages of the element fields of the VTK output (Belytschko law)."""
        x = self.u[:, self.conn]
        R = range(3)
        out = torch.zeros(self.conn.shape[1], 21, dtype=torch.float64, device=self.dev)
        for q in range(len(self.wJ)):
            H = self.grad(x, q)
            F, C, J, P, W = self.stress(H)
            S = [[sum(P[i][k] * F[j][k] for k in R) / J for j in R] for i in R]
            z = torch.zeros_like(J)
            E = [[0.5 * (H[i][j] + H[j][i] + (0.0 if self.law == 3 else sum(H[k][i] * H[k][j] for k in R))) if self.law else z
                  for j in R] for i in R]
            vm = torch.sqrt(0.5 * ((S[0][0] - S[1][1]) ** 2 + (S[1][1] - S[2][2]) ** 2 + (S[2][2] - S[0][0]) ** 2
                                   + 6 * (S[0][1] ** 2 + S[0][2] ** 2 + S[1][2] ** 2)))
            tr, eq = z, z
            if self.law in (1, 2):
                tr = E[0][0] + E[1][1] + E[2][2]
                eq = 0.6666 * torch.sqrt(1.5 * (E[0][0] ** 2 + E[1][1] ** 2 + E[2][2] ** 2)
                                         + 3 * (E[0][1] ** 2 + E[0][2] ** 2 + E[1][2] ** 2))
            out += torch.stack([S[i][j] for i in R for j in R] + [E[i][j] for i in R for j in R] + [vm, tr, eq], 1)
        return (out / len(self.wJ)).cpu().numpy()

    def state(self):
        return [x.reshape(-1).cpu().numpy() for x in (self.u, self.v, self.a)]


def exact(case, seed):
    if case["kind"] == "solve":
        md = box_model(case["nx"], case["ny"], case["nz"], seed, case["elem"] == "tet", case["law"], case["het"])
        if md["mesh"]["n_elem"] * case["steps"] * (1 if case["elem"] == "tet" else 8) > 1.2e9:
            return None
        p = Plain(md, load_list(md) if case["loads"] else None, case["visc"])
        for dst, src in zip((p.u, p.v, p.a), moving_state(md, seed)):
            dst.copy_(torch.as_tensor(src).reshape(3, -1))
        for _ in range(case["steps"]):
            p.step(bool(case["energies"]))
        out = {"state": p.state(), "time": np.array([p.time]), "dt": np.array([p.dt])}
        if case["fields"]:
            out["fields"] = p.fields()
        if case["energies"]:
            h = np.array(p.rows).T
            every = case["energies"]
            for c in (0, 1, 2, 3, 4):  # kept on energy steps only
                h[c][[i for i in range(case["steps"]) if (i + 1) % every]] = np.nan
            out["history"] = list(h)
        return out
    models = [box_model(case["nx"], case["ny"], case["nz"], seed, pull=2e-3)] if case["kind"] == "whole" else \
        cubes(case, seed) if case["kind"] == "batch" else requests(case, seed)
    if sum(m["mesh"]["n_elem"] for m in models) * case["steps"] * 8 > 1.2e9:
        return None
    out = []
    for m in models:
        p = Plain(m)
        for _ in range(case["steps"]):
            p.step()
        out.append(p.state())
    return out[0] if case["kind"] == "whole" else out if case["kind"] == "batch" else [o[0] for o in out]
