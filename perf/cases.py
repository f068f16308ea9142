"""Performance cases: what a user of the framework has it do, over the sizes, element shapes, materials and solver
options of its workloads (``amaru.jl_amd/workloads.py``, ``bench.py`` and the tests).

``listed()`` gives the fixed cases, ``draw(rng)`` more of the same ranges, ``prepare(case, seed)`` what a program holds
before the call (meshed model on the device, targets of the stage), ``run(state)`` one pass through the public entry
points, ``work(case)`` the bytes and operations a pass cannot do without and ``exact(case, seed)`` the same outputs
from plain torch and numpy in 64 bits.

What a pass is, by ``case["call"]``:

* ``step``: one load increment of the device-resident stage driver: ``increment_begin``, ``iters`` Newton-Raphson
  iterations (mount_K, solve_system!, update_state!), ``increment_reject`` (the states go back, so that a pass can be
  repeated) and the increment's displacements and internal forces, for plastic materials also the IP states;
* ``dropin``: the host-vector functions in a row: ``assemble``, ``solve_system``, ``update_state``;
* ``batch``: ``run_analyses`` over independent resident models, pooled;
* ``dynamic``: ``dyn_solve``, a stage of Newmark increments;
* ``output``: ``nodal_values``, the recovery of the output fields at the nodes.
"""
import importlib.util
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package in ``amaru.jl_amd`` (imported as ``amaru_amd``)."""
    if "amaru_amd" not in sys.modules:
        pkg = os.path.join(ROOT, "amaru.jl_amd")
        spec = importlib.util.spec_from_file_location("amaru_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["amaru_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["amaru_amd"]


# ------------------------------------------------------------------ the cases

def _step(name, problem, shape, nips, n, precision="fp64", precond="jacobi", ke="exact", iters=1):
    return dict(name=name, call="step", problem=problem, shape=shape, nips=nips, nx=n[0], ny=n[1], nz=n[2],
                precision=precision, precond=precond, ke=ke, iters=iters)


def listed():
    return [
        # the README's and smoke test's cantilever: 1,500 unknowns, all launches and latency
        _step("cantilever_hex8_small", "cantilever", "HEX8", 8, (20, 4, 4)),
        # an ordinary quadratic model on the defaults of solve(): FP64, Jacobi, exact stiffness; ragged cell counts
        _step("block_hex20_fp64", "block", "HEX20", 27, (17, 19, 15)),
        # the headline block (811,923 DOFs) with the options of the benchmark's step
        _step("block_hex20_headline", "block", "HEX20", 27, (40, 40, 40), "mixed64acc", "two_level", "mfma"),
        # reduced integration and the nodal block preconditioner, a slender quadratic beam
        _step("beam_hex20_reduced", "cantilever", "HEX20", 8, (64, 7, 8), "fp64", "block_jacobi", "mfma"),
        # a served elastic request of tetrahedra near the top of its range (about 180,000 DOFs)
        _step("box_tet10_two_level", "box", "TET10", 4, (49, 12, 13), "mixed64acc", "two_level"),
        # FP32 operator and FP32 accumulation, a served request of HEX8
        _step("box_hex8_mixed", "box", "HEX8", 8, (83, 21, 20), "mixed", "jacobi", "mfma"),
        # the Drucker-Prager footing: a settlement increment with its Newton-Raphson iterations
        _step("footing_dp", "footing", "HEX8", 8, (40, 40, 20), "mixed64acc", "two_level", iters=3),
        # a served von Mises request: prescribed tip deflection beyond first yield
        _step("box_tet10_von_mises", "box_vm", "TET10", 4, (27, 7, 7), "fp64", "two_level", iters=3),
        # mount_K, solve_system! and update_state! on host vectors, one after another
        dict(name="dropin_hex8", call="dropin", problem="box", shape="HEX8", nips=8, nx=57, ny=15, nz=13),
        # independent slender cantilevers solved together (the batched workload, fewer of them)
        dict(name="batch_tet10_cantilevers", call="batch", models=48, cells_lo=500, cells_hi=8000),
        # the dynamic stage solver on a quadratic cantilever
        dict(name="dynamic_hex20", call="dynamic", shape="HEX20", nips=27, nx=31, ny=4, nz=5, nincs=3),
        # output fields at the nodes of a solved quadratic model
        dict(name="nodal_output_hex20", call="output", shape="HEX20", nips=27, nx=21, ny=19, nz=20),
    ]


_RULES = {"HEX8": (8,), "HEX20": (8, 27), "TET10": (4,)}
_DOFS_PER_CELL = {"HEX8": 3.0, "HEX20": 12.0, "TET10": 24.0}


def _cells(rng, shape, dofs, aspect):
    """Ragged cell counts of a box with about ``dofs`` DOFs, ``aspect`` times as many along x."""
    m = (dofs / (_DOFS_PER_CELL[shape] * aspect)) ** (1.0 / 3.0)
    return [max(2, int(round(f * m * rng.uniform(0.85, 1.15)))) for f in (aspect, 1.0, 1.0)]


def draw(rng):
    call = rng.choice(["step"] * 7 + ["dropin", "batch", "dynamic", "output"])
    if call == "batch":
        lo = rng.randint(200, 1500)
        return dict(call="batch", models=rng.randint(5, 48), cells_lo=lo, cells_hi=lo + rng.randint(500, 6000))
    shape = rng.choice(["HEX8", "HEX20", "TET10"])
    nips = rng.choice(_RULES[shape])
    if call == "dynamic":
        # rules that give a regular mass matrix
        shape, nips = rng.choice([("HEX8", 8), ("HEX20", 27)])
        n = _cells(rng, shape, math.exp(rng.uniform(math.log(1e3), math.log(1.5e4))), 6.0)
        return dict(call="dynamic", shape=shape, nips=nips, nx=n[0], ny=n[1], nz=n[2], nincs=rng.randint(2, 4))
    if call == "output":
        shape = rng.choice(["HEX8", "HEX20"])
        n = _cells(rng, shape, math.exp(rng.uniform(math.log(2e3), math.log(1.5e5))), 1.0)
        return dict(call="output", shape=shape, nips=rng.choice(_RULES[shape]), nx=n[0], ny=n[1], nz=n[2])
    if call == "dropin":
        n = _cells(rng, shape, math.exp(rng.uniform(math.log(1e3), math.log(6e4))), 4.0)
        return dict(call="dropin", problem="box", shape=shape, nips=nips, nx=n[0], ny=n[1], nz=n[2])
    problem = rng.choice(["block", "cantilever", "box", "box", "box_vm", "footing"])
    precond = rng.choice(["jacobi", "block_jacobi", "two_level", "two_level"])
    precision = rng.choice(["fp64", "fp64", "mixed64acc", "mixed64acc", "mixed"])
    if problem == "footing":
        shape, nips = "HEX8", 8
        # the footing's loaded strip needs nodes on its edges: cells in fives
        m = rng.randint(2, 7)
        n, iters = [5 * m, 5 * m, rng.randint(4, 3 * m + 2)], 3
    else:
        top = 3e5 if precond == "two_level" else 6e4
        top = min(top, 6e4) if problem in ("cantilever", "box_vm") else top
        aspect = {"block": 1.0, "cantilever": 6.0}.get(problem, 4.0)
        n = _cells(rng, shape, math.exp(rng.uniform(math.log(1e3), math.log(top))), aspect)
        iters = 3 if problem == "box_vm" else 1
    # the matrix-core stiffness takes elastic models and every HEX20 one
    ke = rng.choice(["exact", "mfma"]) if iters == 1 or shape == "HEX20" else "exact"
    return dict(call="step", problem=problem, shape=shape, nips=nips, nx=n[0], ny=n[1], nz=n[2], precision=precision,
                precond=precond, ke=ke, iters=iters)


# ----------------------------------------------------------------- the inputs

def _mesh(am, shape, size, n):
    return am.Mesh(am.Block([[0, 0, 0], list(size)], nx=n[0], ny=n[1], nz=n[2], cellshape=shape))


def _model(case, seed):
    """FEModel (host), boundary conditions and increment size of a case: material constants, box dimensions and loads
    from the seed."""
    am = _package()
    rng = random.Random(seed * 2 + 1)
    u = rng.uniform
    n = (case["nx"], case["ny"], case["nz"])
    problem = case.get("problem", {"dynamic": "cantilever", "output": "block"}.get(case["call"]))
    rho = 0.0
    if problem == "block":
        L = [round(u(0.9, 1.1), 3) for _ in range(3)]
        mat = am.LinearElastic(E=u(25e9, 35e9), nu=u(0.15, 0.25))
        bcs = [("z==0", am.SurfaceBC(ux=0, uy=0, uz=0)),
               (f"z=={L[2]:g}", am.SurfaceBC(tz=-u(0.5e6, 1.5e6), tx=u(-1e5, 1e5)))]
    elif problem == "cantilever":
        L = [round(u(0.9, 1.1), 3), round(u(0.1, 0.13), 3), round(u(0.1, 0.13), 3)]
        mat = am.LinearElastic(E=u(150e9, 210e9), nu=u(0.2, 0.35))
        rho = u(7600.0, 8000.0)
        bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)),
               (f"x=={L[0]:g}", am.SurfaceBC(tz=-u(0.5e5, 1.5e5), ty=u(-3e4, 3e4)))]
    elif problem == "box":
        L = [1.0, round(u(0.23, 0.27), 3), round(u(0.23, 0.27), 3)]
        mat = am.LinearElastic(E=u(70e9, 210e9), nu=u(0.25, 0.33))
        bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==1", am.SurfaceBC(tz=-u(0.5e6, 1.5e6)))]
    elif problem == "box_vm":
        L = [1.0, round(u(0.23, 0.27), 3), round(u(0.23, 0.27), 3)]
        E, fy = u(70e9, 210e9), 250e6
        mat = am.VonMises(E=E, nu=0.3, fy=fy, H=2e9)
        bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)),
               ("x==1", am.SurfaceBC(uz=-u(1.2, 1.8) * 2.0 * fy / (3.0 * E * L[2])))]
    else:
        L = [10.0, 10.0, round(u(4.5, 5.5), 2)]
        mat = am.DruckerPrager(E=u(45e6, 55e6), nu=0.3, alpha=0.23094, kappa=u(22e3, 26e3), H=0.0)
        bcs = [("z==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==0 || x==10", am.SurfaceBC(ux=0)),
               ("y==0 || y==10", am.SurfaceBC(uy=0)),
               (f"z=={L[2]:g} && x>=4 && x<=6 && y>=4 && y<=6", am.NodeBC(uz=-u(0.008, 0.012)))]
    model = am.FEModel(_mesh(am, case["shape"], L, n), [("all", am.MechSolid(rho=rho) if rho else am.MechSolid, mat)],
                       nips=case["nips"])
    model.configure_dofs(bcs)
    return model, bcs


def _batch_models(case, seed):
    """The batched workload's cantilevers: element counts spread over the logarithm between the case's bounds."""
    am = _package()
    rng = random.Random(seed * 2 + 1)
    out = []
    for i in range(case["models"]):
        cells = case["cells_lo"] * (case["cells_hi"] / case["cells_lo"]) ** ((i + 0.5) / case["models"])
        m = max(1, int(round((cells / 60.0) ** (1.0 / 3.0))))
        mesh = _mesh(am, "TET10", (1.0, 0.1, 0.1), (10 * m, m, m))
        model = am.FEModel(mesh, [("all", am.MechSolid, am.LinearElastic(E=rng.uniform(10e9, 200e9),
                                                                         nu=rng.uniform(0.2, 0.35)))])
        load = rng.choice([-1, 1]) * rng.uniform(0.3e3, 1e3)
        bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==1", am.SurfaceBC(tz=load / 0.01))]
        model.configure_dofs(bcs)
        out.append((model, bcs))
    return out


def _output_state(model, seed):
    """IP states of a solved von Mises-free model: smooth stress and strain fields with scatter."""
    rng = np.random.default_rng(seed)
    from_c = model.coords[model.conn].mean(axis=1)
    n = model.ne * model.nips
    st = np.zeros((n, 14))
    X = np.repeat(from_c, model.nips, axis=0)
    for f in range(12):
        a = rng.normal(size=4)
        scale = 1e6 if f < 6 else 1e-4
        st[:, f] = scale * (a[0] + X @ a[1:] + 0.3 * np.sin(3.0 * X[:, f % 3]) + 0.05 * rng.normal(size=n))
    return st


def prepare(case, seed):
    am = _package()
    st = {"case": dict(case)}
    if case["call"] == "batch":
        st["models"] = [(m, b, am.DeviceModel(m)) for m, b in _batch_models(case, seed)]
        for _, _, dev in st["models"]:
            dev.set_coarse()
        return st
    model, bcs = _model(case, seed)
    dev = am.DeviceModel(model)
    st.update(model=model, bcs=bcs, dev=dev)
    if case["call"] == "step":
        U, F = model.bc_vals(bcs)
        st["opts"] = dev.opts(precision=case["precision"], precond=case["precond"])
        dev.set_ke_path(case["ke"])
        if case["precond"] == "two_level":
            dev.set_coarse()
            if case["problem"] == "block":
                dev.set_coarse_refresh("assembly")   # the benchmark forms the coarse operator in every step
        dev.stage_begin(U, F)
    elif case["call"] == "dropin":
        st["U"], st["F"] = model.bc_vals(bcs)
    elif case["call"] == "output":
        dev.state_set(_output_state(model, seed))
    return st


# -------------------------------------------------------------------- a pass

def run(st):
    am = _package()
    case = st["case"]
    call = case["call"]
    if call == "step":
        dev = st["dev"]
        dev.increment_begin(1.0, 1.0, False)
        for it in range(1, case["iters"] + 1):
            r = dev.nr_iteration(it, st["opts"])
            if r["status"] != 0:
                raise RuntimeError(r["message"])
        dU, dF = dev.stage_get(last=True)
        out = {"dU": dU, "dF": dF}
        if case["problem"] in ("box_vm", "footing"):
            out["states"] = dev.state_get()
        dev.increment_reject()
        return out
    if call == "dropin":
        dev = st["dev"]
        U, F = st["U"].copy(), st["F"].copy()
        dev.assemble()
        dev.solve_system(U, F)
        return {"U": U, "F": F, "dFin": dev.update_state(U)}
    if call == "output":
        vals, reps = st["dev"].nodal_values()
        return {"values": [vals[:, i].copy() for i in range(16)], "reps": reps}
    if call == "dynamic":
        from amaru_amd import dynamic as D
        model = st["model"]
        ana = D.DynamicAnalysis(model)
        ana.dev = st["dev"]
        D.addstage(ana, st["bcs"], nincs=case["nincs"], tspan=_tspan(case))
        ok, msg = D.dyn_solve(ana, tol=1.0, alpha=2.0, beta=1e-5)
        if not ok:
            raise RuntimeError(msg)
        return {"u": model.uvals, "f": model.fvals, "v": model.vvals, "a": model.avals}
    from amaru_amd import pool as P
    anas = []
    for model, bcs, dev in st["models"]:
        model.uvals = np.zeros((model.nnodes, 3))
        model.fvals = np.zeros((model.nnodes, 3))
        ana = am.MechAnalysis(model)
        ana.dev = dev
        am.addstage(ana, bcs)
        anas.append(ana)
    for ok, msg in P.run_analyses(anas, npools=3, precision="fp64", precond="two_level"):
        if not ok:
            raise RuntimeError(msg)
    return {"u": np.concatenate([a.model.uvals for a in anas]), "f": np.concatenate([a.model.fvals for a in anas])}


def _tspan(case):
    return 2e-3 * case["nincs"]


# --------------------------------------------------------------------- work

def _counts(case):
    """(nodes, elements, nodes per element, IPs) of a box."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    corners = (nx + 1) * (ny + 1) * (nz + 1)
    if case["shape"] == "HEX8":
        return corners, nx * ny * nz, 8, case["nips"]
    if case["shape"] == "HEX20":
        edges = nx * (ny + 1) * (nz + 1) + (nx + 1) * ny * (nz + 1) + (nx + 1) * (ny + 1) * nz
        return corners + edges, nx * ny * nz, 20, case["nips"]
    return (2 * nx + 1) * (2 * ny + 1) * (2 * nz + 1), 6 * nx * ny * nz, 10, case["nips"]


def work(case):
    """Mesh, targets and states read once, results written once; the operations of the element stiffness
    (sum of B' D B over the IPs) and of the strain and force products.  The linear solve's iterations depend on the
    method and are not counted."""
    if case["call"] == "batch":
        per = math.sqrt(case["cells_lo"] * case["cells_hi"])
        nodes, ne = 1.7 * per, per
        return {"bytes": case["models"] * (nodes * (24 + 48 + 48) + ne * 44 + ne * 4 * 112 * 2),
                "flops": case["models"] * ne * 4 * 2.0 * (6 * 6 * 30 + 6 * 30 * 30)}
    nodes, ne, nn, nq = _counts(case)
    nd = 3 * nn
    mesh = nodes * 24 + ne * (4 * nn + 4)
    if case["call"] == "output":
        return {"bytes": mesh + ne * nq * 96 + nodes * (16 * 8 + 4), "flops": ne * nq * 16 * 2.0 * 7 * 8}
    times = {"step": case.get("iters", 1), "dynamic": case.get("nincs", 1)}.get(case["call"], 1)
    return {"bytes": mesh + nodes * 96 + times * ne * nq * 224,
            "flops": times * ne * nq * 2.0 * (36 * nd + 6 * nd * nd + 4 * 6 * nd)}


# ------------------------------------------- the same in plain torch, 64 bits

_HEX = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1],
                 [0, -1, -1], [1, 0, -1], [0, 1, -1], [-1, 0, -1], [0, -1, 1], [1, 0, 1], [0, 1, 1], [-1, 0, 1],
                 [-1, -1, 0], [1, -1, 0], [1, 1, 0], [-1, 1, 0]], dtype=float)


def _tables(shape, nips):
    """Shape functions (nq, nn), derivatives (nq, nn, 3) and weights at the integration points."""
    if shape == "TET10":
        a, b = (5.0 + 3.0 * math.sqrt(5.0)) / 20.0, (5.0 - math.sqrt(5.0)) / 20.0
        P, w = np.array([[a, b, b], [b, a, b], [b, b, a], [b, b, b]]), np.full(4, 1.0 / 24.0)
    else:
        g, gw = (([-1 / math.sqrt(3), 1 / math.sqrt(3)], [1.0, 1.0]) if nips == 8 else
                 ([-math.sqrt(0.6), 0.0, math.sqrt(0.6)], [5 / 9, 8 / 9, 5 / 9]))
        idx = [(i, j, k) for k in range(len(g)) for j in range(len(g)) for i in range(len(g))]
        P = np.array([[g[i], g[j], g[k]] for i, j, k in idx])
        w = np.array([gw[i] * gw[j] * gw[k] for i, j, k in idx])
    N, D = [], []
    for p in P:
        t = torch.tensor(p, dtype=torch.float64, requires_grad=True)

        def values(t):
            if shape == "TET10":
                L = [1 - t[0] - t[1] - t[2], t[0], t[1], t[2]]
                return torch.stack([x * (2 * x - 1) for x in L] + [4 * L[i] * L[j] for i, j in (
                    (0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3))])
            H = torch.tensor(_HEX[:8 if shape == "HEX8" else 20])
            f = 1 + H * t
            if shape == "HEX8":
                return 0.125 * f.prod(1)
            mid = torch.where(H == 0, 1 - t * t, f).prod(1) * 0.25
            return torch.where((H != 0).all(1), 0.125 * f.prod(1) * ((H * t).sum(1) - 2), mid)

        N.append(values(t).detach().numpy())
        D.append(torch.autograd.functional.jacobian(values, t).numpy())
    return np.array(N), np.array(D), w


class _Elements:
    """Element arrays of a model on the device, Mandel notation: B (ne, nq, 6, nd), weights times determinants."""

    def __init__(self, model, dev):
        self.X = torch.tensor(model.coords, device=dev)
        self.conn = torch.tensor(model.conn.astype(np.int64), device=dev)
        N, D, w = (torch.tensor(a, device=dev) for a in _tables(model.shape, model.nips))
        self.N = N
        C = self.X[self.conn]
        self.ne, self.nn, _ = C.shape
        self.nq, self.nd = len(w), 3 * C.shape[1]
        self.dof = (self.conn[:, :, None] * 3 + torch.arange(3, device=dev)).reshape(self.ne, self.nd)
        self.n = len(self.X) * 3
        self.D_, self.C, self.w = D, C, w

    def gradients(self, e0, e1):
        J = torch.einsum("eai,qaj->eqij", self.C[e0:e1], self.D_)
        G = torch.einsum("qaj,eqjk->eqak", self.D_, torch.linalg.inv(J))
        return G, torch.linalg.det(J) * self.w

    def b_matrix(self, e0, e1):
        G, coef = self.gradients(e0, e1)
        B = torch.zeros(*G.shape[:2], 6, self.nn, 3, dtype=G.dtype, device=G.device)
        x, y, z = G[..., 0], G[..., 1], G[..., 2]
        h = math.sqrt(0.5)
        B[:, :, 0, :, 0], B[:, :, 1, :, 1], B[:, :, 2, :, 2] = x, y, z
        B[:, :, 3, :, 1], B[:, :, 3, :, 2] = h * z, h * y
        B[:, :, 4, :, 0], B[:, :, 4, :, 2] = h * z, h * x
        B[:, :, 5, :, 0], B[:, :, 5, :, 1] = h * y, h * x
        return B.reshape(*G.shape[:2], 6, self.nd), coef

    def chunks(self):
        step = max(1, 40_000_000 // (self.nq * 6 * self.nd))
        return [(e, min(self.ne, e + step)) for e in range(0, self.ne, step)]

    def stiffness(self, D):
        """(ne, nd, nd) of sum B' D B; D (6, 6) or per IP (ne, nq, 6, 6)."""
        out = []
        for a, b in self.chunks():
            B, coef = self.b_matrix(a, b)
            DB = torch.matmul(D if D.dim() == 2 else D[a:b], B) * coef[:, :, None, None]
            m = b - a
            out.append(torch.bmm(B.reshape(m, -1, self.nd).transpose(1, 2).contiguous(), DB.reshape(m, -1, self.nd)))
        return torch.cat(out)

    def mass(self, rho):
        """(ne, nd, nd) of sum rho N' N."""
        coef = torch.cat([self.gradients(a, b)[1] for a, b in self.chunks()]) * rho
        m = torch.einsum("eq,qa,qb->eab", coef, self.N, self.N)
        return torch.einsum("eab,ij->eaibj", m, torch.eye(3, dtype=m.dtype, device=m.device)).reshape(
            self.ne, self.nd, self.nd)

    def strain(self, u):
        return torch.cat([torch.matmul(self.b_matrix(a, b)[0], u[self.dof[a:b]][:, None, :, None])[..., 0]
                          for a, b in self.chunks()])

    def force(self, sig):
        f = torch.zeros(self.n, dtype=sig.dtype, device=sig.device)
        for a, b in self.chunks():
            B, coef = self.b_matrix(a, b)
            fe = torch.matmul(B.transpose(2, 3), (sig[a:b] * coef[:, :, None])[..., None])[..., 0].sum(1)
            f.index_add_(0, self.dof[a:b].reshape(-1), fe.reshape(-1))
        return f

    def product(self, Ke, x):
        y = torch.zeros_like(x)
        return y.index_add_(0, self.dof.reshape(-1), torch.bmm(Ke, x[self.dof][:, :, None]).reshape(-1))

    def diagonal(self, Ke):
        d = torch.zeros(self.n, dtype=Ke.dtype, device=Ke.device)
        return d.index_add_(0, self.dof.reshape(-1), torch.diagonal(Ke, dim1=1, dim2=2).reshape(-1))


def _pcg(apply, diag, free, b, lengths=None):
    """x with apply(x) = b on the free dofs (0 elsewhere); lengths: dofs of independent systems stored one after
    another, each with its own scalars."""
    lengths = torch.tensor([len(b)], device=b.device) if lengths is None else lengths

    def dot(u, v):
        return torch.segment_reduce(u * v, "sum", lengths=lengths) if len(lengths) > 1 else torch.dot(u, v)[None]

    def each(a):
        return torch.repeat_interleave(a, lengths, output_size=len(b)) if len(lengths) > 1 else a

    minv = torch.where(free, 1.0 / diag, torch.zeros_like(diag))
    x = torch.zeros_like(b)
    for tol in (1e-13, 1e-6):   # the second pass refines what the first one left
        r = torch.where(free, b - apply(x), torch.zeros_like(b))
        stop = tol * tol * dot(r, r)
        z = minv * r
        p, rz = z.clone(), dot(r, z)
        for it in range(12000):
            if it % 50 == 0 and bool((dot(r, r) <= stop).all()):
                break
            q = torch.where(free, apply(p), torch.zeros_like(p))
            pq = dot(p, q)
            a = each(torch.where(pq > 0, rz / pq, torch.zeros_like(pq)))
            x, r = x + a * p, r - a * q
            z = minv * r
            rz, old = dot(r, z), rz
            p = z + each(torch.where(old > 0, rz / old, torch.zeros_like(old))) * p
    return x


def _elastic(mat, dev):
    E, nu = mat.E, mat.nu
    c = E / ((1 + nu) * (1 - 2 * nu))
    D = torch.full((6, 6), 0.0, dtype=torch.float64, device=dev)
    D[:3, :3] = c * nu
    D += torch.diag(torch.full((6,), c * (1 - 2 * nu), dtype=torch.float64, device=dev))
    return D


def _dev_parts(s):
    """Deviator of Mandel stresses and its square norm over two (J2)."""
    d = s.clone()
    d[..., :3] -= s[..., :3].mean(-1, keepdim=True)
    return d, 0.5 * (d * d).sum(-1)


def _tangent(mat, De, sig, dlam):
    """(ne, nq, 6, 6) tangents of the IPs at their states."""
    D = De.expand(*sig.shape[:2], 6, 6)
    kind = type(mat).__name__
    if kind == "LinearElastic":
        return De
    s, j2 = _dev_parts(sig)
    nrm = torch.sqrt(2 * j2)[..., None].clamp_min(1e-300)
    one = torch.tensor([1.0, 1.0, 1.0, 0, 0, 0], dtype=sig.dtype, device=sig.device)
    if kind == "VonMises":
        N = V = math.sqrt(1.5) * s / nrm
        hard = math.sqrt(1.5) * mat.H
    else:
        V = mat.alpha * one + s / nrm / math.sqrt(2.0)
        V = torch.where((j2 != 0)[..., None], V, one / math.sqrt(3.0))
        N = V / torch.linalg.norm(V, dim=-1, keepdim=True)
        hard = mat.H
    a, b = N @ De, V @ De
    den = (b * N).sum(-1) + hard
    Dp = D - a[..., :, None] * b[..., None, :] / den[..., None, None]
    return torch.where((dlam != 0)[..., None, None], Dp, D)


def _update(mat, De, de):
    """Stresses and plastic multipliers of a strain increment from the virgin state."""
    tr = de @ De
    kind = type(mat).__name__
    zero = torch.zeros_like(tr[..., 0])
    if kind == "LinearElastic":
        return tr, zero
    s, j2 = _dev_parts(tr)
    sj = torch.sqrt(j2)
    G, K = mat.E / (2 * (1 + mat.nu)), mat.E / (3 * (1 - 2 * mat.nu))
    if kind == "VonMises":
        f = math.sqrt(3.0) * sj - mat.fy
        dl = f / (3 * G + math.sqrt(1.5) * mat.H)
        out = tr - (math.sqrt(6.0) * G * dl / torch.sqrt(2 * j2).clamp_min(1e-300))[..., None] * s
    else:
        j1 = tr[..., :3].sum(-1)
        f = mat.alpha * j1 + sj - mat.kappa
        n = 1 / math.sqrt(3 * mat.alpha ** 2 + 0.5)
        dg = f / (9 * mat.alpha ** 2 * n * K + n * G + mat.H)
        ap = (mat.alpha * j1 - mat.kappa) / (3 * math.sqrt(3.0) * mat.alpha * K + mat.H)
        cone = sj > 0   # the return to the cone is chosen on the previous multiplier, which is zero here
        p1 = (j1 - 9 * dg * mat.alpha * n * K) / 3
        p2 = (j1 - 3 * math.sqrt(3.0) * ap * K) / 3
        dl = torch.where(cone, dg, ap)
        one = torch.tensor([1.0, 1.0, 1.0, 0, 0, 0], dtype=tr.dtype, device=tr.device)
        out = torch.where(cone[..., None], (1 - dg * n * G / sj.clamp_min(1e-300))[..., None] * s +
                          p1[..., None] * one, p2[..., None] * one)
    plastic = f >= 1e-8
    return torch.where(plastic[..., None], out, tr), torch.where(plastic, dl, zero)


def _eq_maps(model, dev):
    """Node-order targets and masks from the model's numbering."""
    eq = torch.tensor(model.eq.reshape(-1).astype(np.int64), device=dev)
    return eq, eq < model.nu


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["call"] == "batch":
        return _exact_batch(case, seed, dev)
    model, bcs = _model(case, seed)
    if case["call"] == "output":
        return _exact_output(model, seed, dev)
    el = _Elements(model, dev)
    mat = model.mats[0]
    De = _elastic(mat, dev)
    eq, free = _eq_maps(model, dev)
    if case["call"] == "dynamic":
        return _exact_dynamic(case, model, bcs, el, De, eq, free)
    Uex, Fex = (torch.tensor(v, device=dev)[eq] for v in model.bc_vals(bcs))
    back = torch.empty_like(eq)
    back[eq] = torch.arange(len(eq), device=dev)
    zero = torch.zeros_like(Uex)
    u, dui, R = zero, torch.where(free, zero, Uex), Fex
    sig = torch.zeros(el.ne, el.nq, 6, dtype=torch.float64, device=dev)
    dlam = sig[..., 0]
    for it in range(case.get("iters", 1)):
        Ke = el.stiffness(_tangent(mat, De, sig, dlam))
        b = R - el.product(Ke, dui)
        dui = dui + _pcg(lambda v: el.product(Ke, v), el.diagonal(Ke), free, b)
        u = u + dui
        sig, dlam = _update(mat, De, el.strain(u))
        F = el.force(sig)
        R = torch.where(free, Fex - F, zero)
        dui = zero
    u, F = u[back].cpu().numpy(), F[back].cpu().numpy()
    if case["call"] == "dropin":
        Fo = model.bc_vals(bcs)[1]
        Fo[model.nu:] = F[model.nu:]
        return {"U": u, "F": Fo, "dFin": F}
    out = {"dU": u, "dF": F}
    if type(mat).__name__ != "LinearElastic":
        eps = el.strain(torch.tensor(u, device=dev)[eq])
        out["states"] = torch.cat([sig, eps, dlam[..., None], dlam[..., None]], dim=-1).reshape(-1, 14).cpu().numpy()
    return out


def _exact_batch(case, seed, dev):
    models = _batch_models(case, seed)
    els = [_Elements(m, dev) for m, _ in models]
    first = np.cumsum([0] + [e.n for e in els])
    Ke = torch.cat([e.stiffness(_elastic(m.mats[0], dev)) for e, (m, _) in zip(els, models)])
    dof = torch.cat([e.dof + int(o) for e, o in zip(els, first)])
    n = int(first[-1])
    lengths = torch.tensor([e.n for e in els], device=dev)

    def product(x):
        return torch.zeros_like(x).index_add_(0, dof.reshape(-1), torch.bmm(Ke, x[dof][:, :, None]).reshape(-1))

    diag = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(
        0, dof.reshape(-1), torch.diagonal(Ke, dim1=1, dim2=2).reshape(-1))
    free = torch.cat([_eq_maps(m, dev)[1] for m, _ in models])
    b = torch.cat([torch.tensor(m.bc_vals(bc)[1], device=dev)[_eq_maps(m, dev)[0]] for m, bc in models])
    x = _pcg(product, diag, free, b, lengths)
    return {"u": x.reshape(-1, 3).cpu().numpy(), "f": product(x).reshape(-1, 3).cpu().numpy()}


def _exact_dynamic(case, model, bcs, el, De, eq, free):
    alpha, beta = 2.0, 1e-5
    K, M = el.stiffness(De), el.mass(float(model.rho[0]))
    F = torch.tensor(model.bc_vals(bcs)[1], device=eq.device)[eq]
    zero = torch.zeros_like(F)
    C = alpha * M + beta * K
    A = _pcg(lambda v: el.product(M, v), el.diagonal(M), free, F)
    V, U = zero, zero
    dt = _tspan(case) / case["nincs"]
    Kp = K + 4 / dt ** 2 * M + 2 / dt * C
    for _ in range(case["nincs"]):
        b = F - el.product(K, U) + el.product(M, A + 4 * V / dt) + el.product(C, V)
        d = _pcg(lambda v: el.product(Kp, v), el.diagonal(Kp), free, b)
        U, V, A = U + d, -V + 2 * d / dt, -A + 4 * (d - V * dt) / dt ** 2
    T = el.product(K, U) + el.product(C, V) + el.product(M, A)
    return {k: v.reshape(-1, 3).cpu().numpy() for k, v in (("u", U), ("f", T), ("v", V), ("a", A))}


def _exact_output(model, seed, dev):
    """Least-squares fits over the eight elements around every inner corner node of the block, averaged per node (in a
    block of two or more cells each way every node belongs to such a patch)."""
    st = _output_state(model, seed)
    h = math.sqrt(0.5)
    s, e = st[:, :6].copy(), st[:, 6:12].copy()
    s[:, 3:] *= h
    e[:, 3:] *= h
    T = s[:, [0, 5, 4, 5, 1, 3, 4, 3, 2]].reshape(-1, 3, 3)
    m = s[:, :3] - s[:, :3].mean(axis=1, keepdims=True)
    vm = np.sqrt(1.5 * (m ** 2).sum(1) + 3.0 * (s[:, 3:] ** 2).sum(1))
    vals = np.concatenate([s, vm[:, None], np.linalg.eigvalsh(T)[:, ::-1], e], axis=1)
    el = _Elements(model, dev)
    nq = model.nips
    ipx = torch.einsum("qa,eai->eqi", el.N, el.C)
    corners = model.conn[:, :8]
    order = np.argsort(corners.reshape(-1), kind="stable")
    nodes, start, cnt = np.unique(corners.reshape(-1)[order], return_index=True, return_counts=True)
    inner = cnt == 8
    elems = torch.tensor(order[start[inner][:, None] + np.arange(8)] // 8, device=dev)   # (patches, 8)
    centre = el.X[torch.tensor(nodes[inner].astype(np.int64), device=dev)]
    v = torch.tensor(vals, device=dev).reshape(model.ne, nq, 16)
    total = torch.zeros(model.nnodes, 16, dtype=torch.float64, device=dev)
    reps = torch.zeros(model.nnodes, dtype=torch.int64, device=dev)
    size = (el.C.amax(dim=(0, 1)) - el.C.amin(dim=(0, 1))) / torch.tensor([8.0], device=dev, dtype=torch.float64)

    def basis(X):
        x, y, z = X[..., 0], X[..., 1], X[..., 2]
        return torch.stack([torch.ones_like(x), x, y, z, x * y, y * z, x * z], dim=-1)

    for a in range(0, len(elems), 4000):
        p = elems[a:a + 4000]
        c = centre[a:a + 4000][:, None, :]
        A = basis((ipx[p].reshape(len(p), -1, 3) - c) / size)
        Q, Rm = torch.linalg.qr(A)
        coef = torch.linalg.solve_triangular(Rm, Q.transpose(1, 2) @ v[p].reshape(len(p), -1, 16), upper=True)
        flat = p.shape[0]
        conn = el.conn[p].reshape(flat, -1)
        srt, _ = torch.sort(conn, dim=1)
        keep = torch.ones_like(srt, dtype=torch.bool)
        keep[:, 1:] = srt[:, 1:] != srt[:, :-1]
        w = basis((el.X[srt] - c) / size) @ coef
        total.index_add_(0, srt[keep], w[keep])
        reps.index_add_(0, srt[keep], torch.ones_like(srt[keep]))
    out = (total / reps[:, None]).cpu().numpy()
    return {"values": [out[:, i] for i in range(16)], "reps": None}
