"""Work that a program using this package has it do, as cases that can be timed and compared.

Chorin projection steps (the package's purpose) on channel-with-hole meshes from the DFG size to half a million pressure
nodes, alone, as an ensemble on one mesh and as a block-diagonal batch of uneven meshes; the linear solvers as a program
calls them by themselves; the sparse products.  A pass of a step case restarts the flow from a given velocity (a parameter
study's inner loop): reset, load the velocity, a few time steps, keep velocity and pressure.  A pass of a solver case loads
a right-hand side, solves from zero and keeps the solution.

A context, a stepper or a solver is laid out once per mesh and used for every start or right-hand side, as a program
does; prepare() makes the start or the right-hand side from the seed.

exact() is the same computation element by element in plain torch, in 64 bits, with Jacobi-preconditioned conjugate
gradients down to rounding."""

import functools
import math

import numpy as np
import torch

from nsfem_amd import cu, fem, mesher

# ---------------------------------------------------------------- the cases


def _step(name, nodes, velocity, pressure, inverse, start, captured=False, instances=1, systems=1, mesh="channel", steps=4):
    return {"name": name, "kind": "step", "mesh": mesh, "nodes": nodes, "velocity": velocity, "pressure": pressure,
            "inverse": inverse, "start": start, "captured": captured, "instances": instances, "systems": systems, "steps": steps}


def listed():
    return [
        # the DFG channel at the size of the coarse mesh in tests/golden (1,890 nodes), every default: what a first run does
        _step("step-dfg-2k", 1890, "pcg", "pcg", False, "zero", mesh="dfg"),
        # the finer of those meshes (10,762 nodes), mixed precision, steps captured as graphs: long runs on a small mesh
        _step("step-dfg-11k-captured", 10762, "pcg_mixed", "amg_pcg_mixed", True, "extrapolate", captured=True, mesh="dfg"),
        # the plain FP64 path: symmetric Gauss-Seidel velocity solves from zero, AMG pressure
        _step("step-60k-fp64", 60013, "pcg", "amg_pcg", False, "zero"),
        # the bench's headline: half a million pressure nodes, two million velocity nodes a component
        _step("step-500k-mixed", 500000, "pcg_mixed", "amg_pcg_mixed", True, "extrapolate"),
        # a parameter sweep on one mesh: eight flows share every matrix
        _step("ensemble-8x40k", 40000, "pcg_mixed", "amg_pcg_mixed", True, "extrapolate", instances=8),
        # uneven meshes in one block-diagonal batch, each step one graph, FP64
        _step("batch-9x25k", 25000, "pcg", "pcg", True, "zero", captured=True, systems=9),
        # a pure-Neumann Poisson solve, AMG-preconditioned, mixed precision
        {"name": "poisson-250k-amg", "kind": "poisson", "nodes": 250000, "method": "amg_pcg_mixed", "columns": 1},
        # the same kind of system for a tile of right-hand sides, independent columns
        {"name": "poisson-100kx16-amg", "kind": "poisson", "nodes": 100003, "method": "amg_pcg_mixed", "columns": 16},
        # and as one block Krylov space
        {"name": "poisson-30kx8-block", "kind": "poisson", "nodes": 30011, "method": "bpcg_mixed", "columns": 8},
        # multicolour Gauss-Seidel in FP32 with its absolute stop, on a velocity mass matrix: the reference's own solver
        {"name": "mass-25k-gs-f32", "kind": "mass", "nodes": 25000, "method": "gs", "f32": True},
        # one product with two columns, P2 pattern, FP64
        {"name": "spmm-p2-250k-f64", "kind": "product", "nodes": 250000, "matrix": "velocityStiffness", "columns": 2, "f32": False},
        # the smallest call: one divergence product on a small mesh, FP32
        {"name": "spmv-div-2k-f32", "kind": "product", "nodes": 2000, "matrix": "velocityPressureDiv", "columns": 1, "f32": True},
    ]


def draw(rng):
    def nodes(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "step", "ensemble", "batch", "poisson", "tile", "mass", "product"])
    mixed = rng.random() < 0.5
    mix = "_mixed" if mixed else ""
    if kind == "step":
        c = _step("", nodes(1500, 250000), "pcg" + mix, "amg_pcg" + mix, rng.random() < 0.6, rng.choice(["zero", "extrapolate"]),
                  captured=rng.random() < 0.3, mesh=rng.choice(["channel", "dfg"]))
    elif kind == "ensemble":
        k = rng.choice([2, 4, 8])
        c = _step("", nodes(2000, 240000 // k), "pcg" + mix, "amg_pcg" + mix, rng.random() < 0.6, rng.choice(["zero", "extrapolate"]),
                  instances=k)
    elif kind == "batch":
        k = rng.randint(2, 9)
        c = _step("", nodes(2000, 20000), "pcg" + mix, "pcg" + mix, rng.random() < 0.6, "zero", captured=rng.random() < 0.5, systems=k)
    elif kind == "poisson":
        return {"kind": "poisson", "nodes": nodes(2000, 250000), "method": "amg_pcg" + mix, "columns": 1}
    elif kind == "tile":
        k = rng.choice([4, 8, 16])
        block = rng.random() < 0.4
        return {"kind": "poisson", "nodes": nodes(2000, 30000 if block else 100000), "method": ("bpcg" if block else "amg_pcg") + mix, "columns": k}
    elif kind == "mass":
        return {"kind": "mass", "nodes": nodes(1000, 60000), "method": rng.choice(["gs", "pcg"]), "f32": rng.random() < 0.5}
    else:
        return {"kind": "product", "nodes": nodes(1000, 250000), "matrix": rng.choice(["velocityStiffness", "pressureStiffness", "velocityPressureDiv", "pressureVelocityDiv"]),
                "columns": rng.choice([1, 2, 3]), "f32": rng.random() < 0.5}
    del c["name"]
    return c


def _p1_entries(v):
    return 7.0 * v


def _p2_entries(v):
    return 50.0 * v  # about 4 v rows of 12.5


def work(case):
    """Every matrix that the pass needs read once per solve or product, every vector read and written once.  Half of a
    batch's largest mesh is about its mean."""
    v = float(case["nodes"])
    if case["kind"] == "step":
        b = case["instances"]
        if case["systems"] > 1:
            v *= 0.5 * case["systems"]
        # convection: 2 v elements of 64 bytes and nu K once per flow; two mass solves, one pressure solve, two divergence products
        matrices = 12 * (2 * _p2_entries(v) + _p1_entries(v) + 2 * 38 * v)
        flow = 64 * 2 * v + 8 * _p2_entries(v) + 8 * 2 * (8 * v + v)
        flops = 2 * b * (2 * 2 * _p2_entries(v) + _p1_entries(v) + 2 * 38 * v) + b * 2 * v * 36 * 24
        return {"bytes": case["steps"] * (matrices + b * flow), "flops": case["steps"] * flops}
    size = 4 if case.get("f32") else 8
    if case["kind"] == "poisson":
        k = case["columns"]
        return {"bytes": (size + 4) * _p1_entries(v) + 2 * size * k * v, "flops": 2 * k * _p1_entries(v)}
    if case["kind"] == "mass":
        return {"bytes": (size + 4) * _p2_entries(v) + 2 * size * 2 * 4 * v, "flops": 4 * _p2_entries(v)}
    k = case["columns"]
    entries, rows, cols = {"velocityStiffness": (_p2_entries(v), 4 * v, 4 * v), "pressureStiffness": (_p1_entries(v), v, v),
                           "velocityPressureDiv": (38 * v, v, 8 * v), "pressureVelocityDiv": (38 * v, 8 * v, v)}[case["matrix"]]
    return {"bytes": (size + 4) * entries + 4 * rows + size * k * (rows + cols), "flops": 2 * k * entries}


def tolerance(case):
    """About four times the distance from exact() that the largest case of a kind shows."""
    if case["kind"] == "product":
        return {"rel": 5e-7} if case["f32"] else {"rel": 1e-15, "max": 1e-13}
    if case["kind"] == "mass":
        return {"rel": 5e-6} if case["f32"] else {"rel": 1e-9}
    if case["kind"] == "poisson":
        return {"rel": 5e-10}  # residuals of 1e-10; block solves come closest to it
    return {"rel": 2e-8}  # solves to 1e-10: the pressure's condition number at half a million nodes


# ------------------------------------------------- meshes, contexts, handles


def _peak(case):
    return 1.0 if case.get("mesh") == "dfg" else 1.5


def _height(case):
    return 0.41 if case.get("mesh") == "dfg" else 1.0


def _viscosity(case):
    return 1e-3 if case.get("mesh") == "dfg" else 2.4e-3


def _sizes(case):
    k = case["systems"]
    return [int(round(case["nodes"] * 0.2 ** (i / max(1, k - 1)))) for i in range(k)]


@functools.lru_cache(maxsize=64)
def _mesh(kind, nodes, seed=20241103):
    m = mesher.dfg_channel(nodes, seed=seed) if kind == "dfg" else mesher.channel_mesh(nodes, seed=seed)
    return mesher.to_triangle_mesh(m), float(m["h"])


@functools.lru_cache(maxsize=64)
def _context(kind, nodes, systems):
    case = {"mesh": kind, "nodes": nodes, "systems": systems}
    cond = fem.DfgConditions(viscosity=_viscosity(case), peakVelocity=_peak(case), channelHeight=_height(case))
    if systems == 1:
        return fem.ChorinContext(_mesh(kind, nodes)[0], cond, gpu_assembly=True)
    return fem.ChorinContext.batch([_mesh(kind, n, 20241103 + i)[0] for i, n in enumerate(_sizes(case))], [cond] * systems,
                                   gpu_assembly=True)


@functools.lru_cache(maxsize=64)
def _parts(kind, nodes, systems):
    """A batch's meshes as contexts of their own."""
    case = {"mesh": kind, "nodes": nodes, "systems": systems}
    cond = fem.DfgConditions(viscosity=_viscosity(case), peakVelocity=_peak(case), channelHeight=_height(case))
    return [fem.ChorinContext(_mesh(kind, n, 20241103 + i)[0], cond, gpu_assembly=True) for i, n in enumerate(_sizes(case))]


def _tau(case):
    """A time step inside the explicit scheme's limit (which is about h^2 / (270 nu) on these meshes)."""
    h = min(_mesh(case["mesh"], n, 20241103 + i)[1] for i, n in enumerate(_sizes(case)))
    return h * h / (700 * _viscosity(case))


def _inflow_scale(case):
    return [1.0 - 0.4 * b / case["instances"] for b in range(case["instances"])]


_handles = {}


def _stepper(case):
    key = repr(sorted((k, v) for k, v in case.items() if k not in ("name", "steps")))
    if key not in _handles:
        ctx = _context(case["mesh"], case["nodes"], case["systems"])
        extra = case["start"] == "extrapolate"
        cfg = fem.ChorinConfig(fem.SolverConfig(case["velocity"], 500, 1e-10, 1), fem.SolverConfig(case["pressure"], 6000, 1e-10, 1),
                               stepGraph=int(case["captured"]),
                               pressureStart=fem.PRESSURE_START_EXTRAPOLATE if extra else fem.PRESSURE_START_LAST,
                               velocityStart=fem.VELOCITY_START_EXTRAPOLATE if extra else fem.VELOCITY_START_ZERO)
        ch = fem.Chorin(ctx, cfg, instances=case["instances"], inflow_scale=_inflow_scale(case) if case["instances"] > 1 else None)
        if case["inverse"]:
            ch.set_solver_option("preconditioner", 1, "velocity")
            if case["systems"] > 1:
                ch.set_solver_option("preconditioner", 1, "pressure")
        ch.set_time_step(_tau(case))
        _handles[key] = ch
    return _handles[key]


_MATRIX = {"poisson": "pressureStiffness", "mass": "velocityMass"}


def _solver(case):
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _handles:
        m = _context("channel", case["nodes"], 1).matrix(_MATRIX[case["kind"]])
        arrays = (m[0], m[2], m[3], m[4])
        if case["kind"] == "poisson":
            s = cu.createSolver(case["method"], case["columns"], arrays, 6000, 1e-10, 1, dtype=np.float64)
            s.setOption("projectMean", 1)
        else:
            # the reference's stop is an absolute residual; a mass matrix row is about h^2 / 3
            target = (1e-6 if case["f32"] else 1e-10) * (_mesh("channel", case["nodes"])[1] ** 2 if case["method"] == "gs" else 1)
            s = cu.createSolver(case["method"], 2, arrays, 200, target, 1, dtype=np.float32 if case["f32"] else np.float64)
        _handles[key] = s
    return _handles[key]


def _matrix(case):
    key = repr(sorted((k, v) for k, v in case.items() if k not in ("name", "columns")))
    if key not in _handles:
        m = _context("channel", case["nodes"], 1).matrix(case["matrix"])
        _handles[key] = cu.csrF(*m, dtype=np.float32 if case["f32"] else np.float64)
    return _handles[key]


# ------------------------------------------------------------------- inputs


def _start_velocity(case, seed):
    """The inflow's parabola along the channel, smooth seeded eddies of some per cent and a seeded perturbation of 1e-3, on the
    CPU in 64 bits (flow after flow for an ensemble, all x and then all y components for a batch)."""
    parts = _parts(case["mesh"], case["nodes"], case["systems"]) if case["systems"] > 1 else [_context(case["mesh"], case["nodes"], 1)]
    xy = torch.cat([torch.from_numpy(c.velocity_mesh()[0]) for c in parts])
    h = _height(case)
    x, y = xy[:, 0], xy[:, 1]
    g = torch.Generator().manual_seed(seed)
    flows = []
    for scale in _inflow_scale(case):
        ux = scale * _peak(case) * y * (h - y) / (h * h)
        uy = torch.zeros_like(ux)
        for k in range(1, 4):
            a, b = torch.rand(2, generator=g, dtype=torch.float64) * 0.02 * _peak(case)
            t, s = torch.rand(2, generator=g, dtype=torch.float64) * 2 * math.pi
            wall = y * (h - y) * 4 / (h * h)
            ux = ux + a * wall * torch.sin(k * 2 * math.pi * x / (2 * h) + t)
            uy = uy + b * wall * torch.sin(k * 2 * math.pi * x / (2 * h) + s)
        u = torch.cat([ux, uy])
        flows.append(u + 1e-3 * _peak(case) * torch.randn(u.shape, generator=g, dtype=torch.float64))
    return torch.cat(flows)


def _right_hand_side(case, seed):
    """columns x n on the CPU in 64 bits: uniform in [-1, 1], of zero mean for the Neumann systems; a mass system's is the mass
    matrix' scale of a velocity."""
    g = torch.Generator().manual_seed(seed)
    ctx = _context("channel", case["nodes"], 1)
    if case["kind"] == "poisson":
        b = torch.rand((case["columns"], ctx.numPressureNodes), generator=g, dtype=torch.float64) * 2 - 1
        return b - b.mean(dim=1, keepdim=True)
    b = torch.rand((2, ctx.numVelocityNodes), generator=g, dtype=torch.float64) * 2 - 1
    b = b * _mesh("channel", case["nodes"])[1] ** 2
    return b.float().double() if case["f32"] else b


def _operand(case, seed):
    rows, cols = _matrix(case).rows, _matrix(case).cols
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((case["columns"], cols), generator=g, dtype=torch.float64)
    return x.float().double() if case["f32"] else x


def _view(t):
    return cu.vec.view(t.data_ptr(), t.numel(), np.float32 if t.dtype == torch.float32 else np.float64, owner=t)


def prepare(case, seed):
    if case["kind"] == "step":
        ch = _stepper(case)
        ctx = ch.ctx
        n, v = 2 * ctx.numVelocityNodes * case["instances"], ctx.numPressureNodes * case["instances"]
        start = _start_velocity(case, seed).cuda()
        u, p = (torch.zeros(k, dtype=torch.float64, device="cuda") for k in (n, v))
        pu, pp = ch.state_pointers()
        state = {"ch": ch, "steps": case["steps"], "out": (u, p), "load": (_view(start), cu.vec.view(pu, n, np.float64, owner=ch)),
                 "keep": ((cu.vec.view(pu, n, np.float64, owner=ch), _view(u)), (cu.vec.view(pp, v, np.float64, owner=ch), _view(p)))}
    elif case["kind"] == "product":
        m = _matrix(case)
        x = _operand(case, seed).to(torch.float32 if case["f32"] else torch.float64).cuda()
        y = torch.zeros((case["columns"], m.rows), dtype=x.dtype, device="cuda")
        product = cu.spmv(m) if case["columns"] == 1 else cu.spmm(m, case["columns"])
        state = {"product": product, "x": _view(x), "y": _view(y), "out": y}
    else:
        s = _solver(case)
        b = _right_hand_side(case, seed).to(torch.float32 if case.get("f32") else torch.float64).cuda()
        x = torch.zeros_like(b)
        state = {"solver": s, "b": _view(b), "x": _view(x), "out": x}
    torch.cuda.synchronize()  # the package has a stream of its own
    return state


def run(state):
    if "ch" in state:
        ch = state["ch"]
        ch.reset()
        state["load"][0].copyTo(state["load"][1])
        for _ in range(state["steps"]):
            ch.step()
        for source, to in state["keep"]:
            source.copyTo(to)
    elif "product" in state:
        state["product"].compute(state["x"], state["y"])
    else:
        s = state["solver"]
        state["b"].copyTo(s.getRhs())
        s.getSol().memsetZero()
        s.solve()
        s.getSol().copyTo(state["x"])
    return state["out"]


# -------------------------------------------- the same in 64 bits, in torch

_A, _B = 0.445948490915965, 0.091576213509771
_WA, _WB = 0.223381589678011 / 2, 0.109951743655322 / 2
_POINTS = [(_A, _A, _WA), (1 - 2 * _A, _A, _WA), (_A, 1 - 2 * _A, _WA), (_B, _B, _WB), (1 - 2 * _B, _B, _WB), (_B, 1 - 2 * _B, _WB)]


def _quadratic(x, y):
    """Values and both derivatives of the six quadratic shape functions: corners 0, 2, 4, the sides' middles 1, 3, 5."""
    l0 = 1 - x - y
    f = [l0 * (2 * l0 - 1), 4 * x * l0, x * (2 * x - 1), 4 * x * y, y * (2 * y - 1), 4 * y * l0]
    fx = [1 - 4 * l0, 4 * (l0 - x), 4 * x - 1, 4 * y, 0.0, -4 * y]
    fy = [1 - 4 * l0, -4 * x, 0.0, 4 * x, 4 * y - 1, 4 * (l0 - y)]
    return f, fx, fy


def _linear(x, y):
    return [1 - x - y, x, y], [-1.0, 1.0, 0.0], [-1.0, 0.0, 1.0]


class _Elements:
    """One mesh's integrals; a product gathers an element's values, applies its small matrix and adds the result up."""

    def __init__(self, xy, el, el1, device):
        self.el, self.el1 = (torch.from_numpy(e.astype(np.int64)).to(device) for e in (el, el1))
        xy = torch.from_numpy(xy).to(device)
        self.n, self.v = len(xy), int(el1.max()) + 1
        p0, p1, p2 = (xy[self.el[:, k]] for k in (0, 2, 4))
        a, b = p1 - p0, p2 - p0
        det = a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]
        # rows: the reference coordinates' gradients
        inv = torch.stack([torch.stack([b[:, 1], -b[:, 0]], 1), torch.stack([-a[:, 1], a[:, 0]], 1)], 1) / det[:, None, None]
        self.w = det.abs()[:, None] * torch.tensor([p[2] for p in _POINTS], dtype=torch.float64, device=device)

        def at(shape):
            f, fx, fy = torch.tensor([shape(x, y) for x, y, _ in _POINTS], dtype=torch.float64, device=device).unbind(1)
            fx, fy = fx[None, :, None, :], fy[None, :, None, :]
            return f, fx * inv[:, 0][:, None, :, None] + fy * inv[:, 1][:, None, :, None]

        self.f2, self.g2 = at(_quadratic)  # (q, 6) and (e, q, 2, 6)
        self.f1, self.g1 = at(_linear)

    def matrix(self, local, el, n):
        k = el.shape[1]
        r, c = el[:, :, None].expand(-1, k, k).reshape(-1), el[:, None, :].expand(-1, k, k).reshape(-1)
        return torch.sparse_coo_tensor(torch.stack([r, c]), local.reshape(-1), (n, n)).coalesce().to_sparse_csr()

    def mass(self):
        return self.matrix(torch.einsum("eq,qi,qj->eij", self.w, self.f2, self.f2), self.el, self.n)

    def stiffness(self, order):
        g, el, n = (self.g2, self.el, self.n) if order == 2 else (self.g1, self.el1, self.v)
        return self.matrix(sum(torch.einsum("e,ei,ej->eij", self.w[:, q], g[:, q, d], g[:, q, d]) for q in range(len(_POINTS)) for d in range(2)), el, n)

    def add(self, local, el, n):
        return torch.zeros(n, dtype=torch.float64, device=local.device).index_add_(0, el.reshape(-1), local.reshape(-1))

    def advance(self, u, nu):
        """(nu K + C(u)) u, both components."""
        out = []
        vel = [u[d][self.el] for d in range(2)]
        flow = [v @ self.f2.T for v in vel]
        for d in range(2):
            grad = [torch.einsum("eqi,ei->eq", self.g2[:, :, c], vel[d]) for c in range(2)]
            local = torch.einsum("eq,qi->ei", self.w * (flow[0] * grad[0] + flow[1] * grad[1]), self.f2)
            local = local + nu * sum(torch.einsum("eq,eqi->ei", self.w * grad[c], self.g2[:, :, c]) for c in range(2))
            out.append(self.add(local, self.el, self.n))
        return out

    def divergence(self, u):
        d = sum(torch.einsum("eqi,ei->eq", self.g2[:, :, c], u[c][self.el]) for c in range(2))
        return self.add(torch.einsum("eq,qi->ei", self.w * d, self.f1), self.el1, self.v)

    def gradient(self, p):
        return [self.add(torch.einsum("eq,qi->ei", self.w * torch.einsum("eqi,ei->eq", self.g1[:, :, c], p[self.el1]), self.f2), self.el, self.n)
                for c in range(2)]


def _conjugate_gradients(a, diag, b, free=None, neumann=False, tol=1e-14, most=20000):
    """a x = b for the columns of b (n x k); `free`: the rows that are solved for, the others stay zero."""
    if free is not None:
        b = b * free[:, None]
    inv = (1 / diag)[:, None]
    x, r = torch.zeros_like(b), b.clone()
    z = inv * r
    p, rz = z.clone(), (r * z).sum(0)
    stop = tol * b.norm(dim=0)
    for it in range(most):
        q = a @ p
        if free is not None:
            q = q * free[:, None]
        pq = (p * q).sum(0)
        alpha = torch.where(pq > 0, rz / pq, torch.zeros_like(rz))
        x, r = x + alpha * p, r - alpha * q
        if neumann:
            r = r - r.mean(0)
        if it % 25 == 24 and bool((r.norm(dim=0) <= stop).all()):
            break
        z = inv * r
        new = (r * z).sum(0)
        p = z + torch.where(rz > 0, new / rz, torch.zeros_like(rz)) * p
        rz = new
    return x - x.mean(0) if neumann else x


def _diagonal(a):
    n = a.shape[0]
    row = torch.repeat_interleave(torch.arange(n, device=a.device), a.crow_indices().diff())
    on = row == a.col_indices()
    return torch.zeros(n, dtype=torch.float64, device=a.device).index_add_(0, row[on], a.values()[on])


def _exact_steps(case, context, u, scale, tau, device):
    e = _Elements(context.velocity_mesh()[0], context.velocity_mesh()[1], context.pressure_mesh()[1], device)
    ids = [torch.from_numpy(context.dirichlet(k)[0].astype(np.int64)).to(device) for k in ("vx", "vy")]
    values = [scale * torch.from_numpy(context.dirichlet(k)[1]).to(device) for k in ("vx", "vy")]
    free = torch.zeros(e.v, dtype=torch.float64, device=device)
    free[torch.from_numpy(context.internal_pressure().astype(np.int64)).to(device)] = 1
    m, k = e.mass(), e.stiffness(1)
    dm, dk = _diagonal(m), _diagonal(k)
    u = [c.to(device).clone() for c in u]
    p = torch.zeros(e.v, dtype=torch.float64, device=device)

    def correct(rhs):
        a = _conjugate_gradients(m, dm, torch.stack(rhs, 1))
        for d in range(2):
            u[d] = u[d] - tau * a[:, d]
            u[d][ids[d]] = values[d]

    for _ in range(case["steps"]):
        correct(e.advance(u, _viscosity(case)))
        p = _conjugate_gradients(k, dk, -e.divergence(u)[:, None] / tau, free)[:, 0]
        correct(e.gradient(p))
    return u, p


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "product":
        m = _context("channel", case["nodes"], 1).matrix(case["matrix"])
        values = torch.from_numpy(m[4].astype(np.float32).astype(np.float64) if case["f32"] else m[4])
        row = torch.repeat_interleave(torch.arange(m[0]), torch.from_numpy(m[2].astype(np.int64)).diff())
        x = _operand(case, seed)[:, torch.from_numpy(m[3].astype(np.int64))] * values
        return torch.zeros((case["columns"], m[0]), dtype=torch.float64).index_add_(1, row, x)
    if case["kind"] != "step":
        c = _context("channel", case["nodes"], 1)
        e = _Elements(c.velocity_mesh()[0], c.velocity_mesh()[1], c.pressure_mesh()[1], device)
        a = e.stiffness(1) if case["kind"] == "poisson" else e.mass()
        b = _right_hand_side(case, seed).to(device)
        return _conjugate_gradients(a, _diagonal(a), b.T.contiguous(), neumann=case["kind"] == "poisson").T.contiguous()
    u = _start_velocity(case, seed)
    tau = _tau(case)
    if case["systems"] == 1:
        c = _context(case["mesh"], case["nodes"], 1)
        flows = u.reshape(case["instances"], 2, -1)
        got = [_exact_steps(case, c, [f[0], f[1]], s, tau, device) for f, s in zip(flows, _inflow_scale(case))]
        return torch.cat([torch.cat(g[0]) for g in got]), torch.cat([g[1] for g in got])
    parts, at = [], 0
    flow = u.reshape(2, -1)
    for c in _parts(case["mesh"], case["nodes"], case["systems"]):
        own = flow[:, at:at + c.numVelocityNodes]
        at += c.numVelocityNodes
        parts.append(_exact_steps(case, c, [own[0], own[1]], 1.0, tau, device))
    return torch.cat([torch.cat([g[0][d] for g in parts]) for d in range(2)]), torch.cat([g[1] for g in parts])
