"""Workloads that time this library as its users call it.

Each case is one pass through the public entry points of ``sonium_amd``: the
dense Burton-Miller assembly (rigid bodies, mixed boundary conditions and
parameter derivatives), FP64 products and Krylov solves, low-precision
refinement, batches and sweeps, field evaluation and the training of the
warm-start network.  ``exact`` restates the mathematics in plain FP64 torch:
the 13-point panel rule with its near-pair subdivision, the self-panel rules,
the incident field, the 7-point field rule and the network.

Sizes follow the benchmark and test configurations: spheres of 320 to 20480
panels, 1 to 64 right-hand sides, batches of uneven ellipsoids, groups of
equally spaced wavenumbers, 16384-sample training steps.
"""

import functools
import math

import numpy as np
import torch

import sonium_amd as sa
from sonium_amd import mesh as meshes
from sonium_amd import warmstart

MAX_PANELS = 20480


@functools.lru_cache(maxsize=None)
def context():
    """One context per process, as a user's program keeps."""
    return sa.Context(0)


# --------------------------------------------------------------------------
# The cases


def listed():
    return [
        # The smallest whole job: a 320-panel sphere assembled and solved for one plane wave with
        # host vectors, as a script or an optimiser calls it.  Launches and host latency.
        {"name": "solve_320", "kind": "solve", "n_theta": 9, "n_phi": 20, "k": 1.0, "restart": 50},
        # The operator assembly of one frequency at the single-GPU scale of the benchmark.
        {"name": "assemble_20480", "kind": "assemble", "n_theta": 65, "n_phi": 160, "k": 10.0},
        # An absorber optimisation: pressure, admittance and vibrating panels, the system and its
        # wavenumber derivative, on a mesh whose panel count is no multiple of any tile.
        {"name": "derivative_4378", "kind": "derivative", "n_theta": 12, "n_phi": 199, "k": 5.0},
        # The plain solve of that assembled system: restarted GMRES, vectors on the device.
        {"name": "gmres_20480", "kind": "gmres", "n_theta": 65, "n_phi": 160, "k": 10.0, "restart": 100},
        # The FP64 block product behind every many-right-hand-side solver.
        {"name": "product_10240x64", "kind": "product", "n_theta": 65, "n_phi": 80, "k": 7.0, "columns": 64},
        # solve_many: many incident directions on one body (head-related transfer functions).
        {"name": "solve_many_5056x24", "kind": "solve_many", "n_theta": 33, "n_phi": 79, "k": 5.0, "columns": 24,
         "restart": 30},
        # One frequency in the chosen mixed-precision form: assembly, FP16 copy, refinement, one wave.
        {"name": "refine_20480", "kind": "refine", "n_theta": 65, "n_phi": 160, "k": 10.0, "columns": 1,
         "format": "fp16"},
        # The same form with 64 directions and BF16 storage.
        {"name": "refine_10240x64", "kind": "refine", "n_theta": 65, "n_phi": 80, "k": 7.0, "columns": 64,
         "format": "bf16"},
        # Many uneven scatterers at once: 24 ellipsoids of 320 to 5120 panels, 1 to 16 directions each.
        {"name": "batch_24", "kind": "batch", "instances": 24, "level_max": 4, "format": "fp16_ir"},
        # One group of a frequency sweep on one body, started from the network's guesses.
        {"name": "sweep_5120x16", "kind": "sweep", "n_theta": 33, "n_phi": 80, "k": 4.0, "dk": 0.11, "instances": 16,
         "width": 512},
        # The pressure around a solved body on an observation grid.
        {"name": "field_5000", "kind": "field", "n_theta": 65, "n_phi": 80, "k": 7.0, "points": 5000,
         "velocity": True},
        # Training the warm-start network on solver solutions, its batch size and width.
        {"name": "train_16384", "kind": "train", "width": 512, "batch": 16384, "steps": 40, "samples": 400000},
    ]


def _sphere_size(rng, lo, hi):
    """(n_theta, n_phi) of a Fibonacci sphere with about lo..hi panels, spread over the logarithm."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n_theta = rng.randint(5, max(5, min(70, int(target / 40))))
    n_phi = int(target / (2 * (n_theta - 1)))
    while 2 * (n_theta - 1) * n_phi > hi:
        n_phi -= 1
    return n_theta, max(3, n_phi)


def _wavenumber(rng, n_theta, n_phi, lo=0.05, hi=0.9):
    """A wavenumber that the mesh resolves: k times the panel edge in lo..hi."""
    panels = 2 * (n_theta - 1) * n_phi
    edge = math.sqrt(4 * math.pi / panels * 4 / math.sqrt(3))
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / edge, 4)


def draw(rng):
    kind = rng.choice(["solve", "assemble", "derivative", "gmres", "product", "solve_many", "refine", "batch",
                       "sweep", "field", "train"])
    c = {"kind": kind}
    if kind == "batch":
        c.update(instances=rng.randint(2, 24), level_max=rng.choice([2, 3, 3, 4]),
                 format=rng.choice(["fp16_ir", "fp16_ir", "bf16_ir", "fp64"]))
        return c
    if kind == "train":
        c.update(width=rng.choice([64, 128, 256, 512]), batch=256 * int(math.exp(rng.uniform(0, math.log(64)))),
                 steps=rng.randint(2, 40), samples=rng.randint(5000, 400000))
        return c
    top = {"solve": 2600, "assemble": MAX_PANELS, "derivative": 6000, "gmres": MAX_PANELS, "product": 10240,
           "solve_many": 5200, "refine": MAX_PANELS, "sweep": 5120, "field": 10240}[kind]
    nt, nphi = _sphere_size(rng, 200, top)
    c.update(n_theta=nt, n_phi=nphi, k=_wavenumber(rng, nt, nphi))
    if kind == "solve":
        c.update(restart=rng.choice([30, 50]))
    elif kind == "gmres":
        c.update(restart=rng.choice([50, 100]))
    elif kind == "product":
        c.update(columns=rng.randint(1, 64))
    elif kind == "solve_many":
        c.update(columns=rng.randint(2, 24), restart=30)
    elif kind == "refine":
        c.update(columns=rng.randint(1, 64) if 2 * (nt - 1) * nphi <= 10240 else 1,
                 format=rng.choice(["fp16", "bf16"]))
    elif kind == "sweep":
        c.update(instances=rng.randint(2, 16), width=rng.choice([128, 256, 512]),
                 dk=round(0.2 * c["k"] / 16 * rng.uniform(0.3, 1.5), 5))
    elif kind == "field":
        c.update(points=int(math.exp(rng.uniform(math.log(3), math.log(5000)))), velocity=rng.random() < 0.5)
    return c


# --------------------------------------------------------------------------
# Inputs


def _rotation(g):
    q, r = np.linalg.qr(g.standard_normal((3, 3)))
    q = q * np.sign(np.diag(r))
    if np.linalg.det(q) < 0:
        q[:, 0] = -q[:, 0]
    return q


@functools.lru_cache(maxsize=8)
def _sphere(n_theta, n_phi):
    return meshes.fibonacci_sphere(1.0, n_theta, n_phi)


def _panels(case):
    return 2 * (case["n_theta"] - 1) * case["n_phi"]


def _inputs(case, seed):
    """What the user has on the host, from the seed alone: mesh, wavenumbers, boundary data, directions."""
    g = np.random.default_rng([20261204, int(seed)])
    kind = case["kind"]
    d = {"rng": g}
    if kind == "train":
        return d
    if kind == "batch":
        d["meshes"], d["ks"], d["dirs"] = [], [], []
        for i in range(case["instances"]):
            # sizes in turn, the largest one third of the instances, so that every seed costs about the same
            level = 2 + i % (case["level_max"] - 1)
            m = meshes.ellipsoid(g.uniform(0.5, 1.5, size=3), level)
            d["meshes"].append(meshes.Mesh(m.nodes @ _rotation(g).T, m.triangles))
            d["ks"].append(float(g.uniform(1.0, {2: 4.0, 3: 6.0, 4: 8.0}[level])))
            d["dirs"].append(meshes.uniform_directions(g, 1 + (5 * i + 3) % 16))
        return d
    base = _sphere(case["n_theta"], case["n_phi"])
    d["mesh"] = meshes.Mesh(base.nodes @ _rotation(g).T * g.uniform(0.95, 1.05), base.triangles)
    d["k"] = case["k"] * float(g.uniform(0.97, 1.03))
    d["dirs"] = meshes.uniform_directions(g, case.get("columns", 1))
    n = d["mesh"].num_elements
    if kind == "derivative":
        u = g.random(n)
        d["bc_type"] = (u < 0.2).astype(np.int32)  # a fifth of the panels with prescribed pressure
        adm = np.full(n, np.nan + 0j)
        absorbing = (u > 0.6) & (d["bc_type"] == 0)
        adm[absorbing] = (g.uniform(0.2, 1.0, n) + 0.2j * g.standard_normal(n))[absorbing] / (1.21 * 343.0)
        d["admittance"] = adm
        value = np.zeros(n, dtype=np.complex128)
        driven = g.choice(n, size=min(n, 12), replace=False)  # a small vibrating patch
        value[driven] = 1e-3 * (g.standard_normal(driven.size) + 1j * g.standard_normal(driven.size))
        d["bc_value"] = value
    if kind == "product":
        d["X"] = g.standard_normal((n, case["columns"])) + 1j * g.standard_normal((n, case["columns"]))
    if kind == "field":
        p = g.standard_normal((case["points"], 3))
        d["points"] = p / np.linalg.norm(p, axis=1, keepdims=True) * g.uniform(1.3, 4.0, (case["points"], 1))
        c, nn, _ = d["mesh"].element_geometry()
        phase = np.exp(1j * d["k"] * (c @ d["dirs"][0]))
        d["p"] = phase * (1.5 + 0.3 * g.standard_normal(n))
        d["v"] = phase * 1e-3 * (1.0 + 0.3 * g.standard_normal(n)) if case["velocity"] else None
    return d


def _he_parameters(g, width):
    out = []
    for rows, cols in ((width, 64), (width, width), (width, width), (2, width)):
        bound = math.sqrt(6.0 / cols) * (0.1 if rows == 2 else 1.0)
        out += [g.uniform(-bound, bound, rows * cols), np.zeros(rows)]
    return np.concatenate(out).astype(np.float32)


def _samples(g, count):
    """Raw samples {centroid, normal, direction, k} of spheres and their phase-free densities (a smooth model)."""
    c = g.standard_normal((count, 3))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    d = meshes.uniform_directions(g, count)
    k = g.uniform(1.0, 12.0, (count, 1))
    raw = np.concatenate([c, c, d, k], axis=1).astype(np.float32)
    mu = np.sum(c * d, axis=1)
    t = np.stack([1.0 - 0.8 * mu + 0.1 * np.cos(k[:, 0] * (1 + mu)), 0.3 * np.sin(k[:, 0] * (1 + mu)) / k[:, 0]], axis=1)
    return raw, t.astype(np.float32)


class _DeviceMemory:
    """A device allocation of the library, described for torch; it keeps the owning object alive."""

    def __init__(self, owner, pointer, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<c16", "data": (int(pointer), False),
                                         "strides": None, "version": 3}


def _view(owner, pointer, shape):
    """A tensor over the library's memory.  A result outlives the state it came from, so the tensor holds the
    owner of its memory."""
    t = torch.as_tensor(_DeviceMemory(owner, pointer, shape), device="cuda")
    assert t.data_ptr() == pointer
    t.owner = owner
    return t


def _system_views(system):
    a, lda, b = system.device_pointers()
    n = system.num_dofs
    assert lda == n  # rows are contiguous
    return _view(system, a, (n, n)), _view(system, b, (n,))


def _device_block(values):
    v = sa.DeviceVector(context(), values.size)
    v.upload(values)
    return v


def prepare(case, seed):
    ctx = context()
    kind = case["kind"]
    d = _inputs(case, seed)
    s = {"case": dict(case), "kind": kind}
    if kind == "train":
        s["parameters"] = _he_parameters(d["rng"], case["width"])
        s["raw"], s["targets"] = _samples(d["rng"], case["samples"])
        return s
    if kind == "batch":
        s["meshes"] = [sa.TbemMesh(ctx, m) for m in d["meshes"]]
        s["batch"] = sa.Batch(ctx, s["meshes"])
        s["batch"].set_problem(d["ks"], d["dirs"])
        return s
    physics = sa.PhysicsParams.from_wavenumber(d["k"])
    s["physics"], s["beta"] = physics, physics.burton_miller_beta()
    if kind == "derivative":
        s["mesh"] = sa.TbemMesh(ctx, d["mesh"], d["bc_type"], d["bc_value"], d["admittance"])
    else:
        s["mesh"] = sa.TbemMesh(ctx, d["mesh"])
    if kind == "field":
        s.update(points=d["points"], p=d["p"], v=d["v"], wave=sa.IncidentField(d["dirs"]))
        return s
    n = d["mesh"].num_elements
    if kind == "sweep":
        count = case["instances"]
        s["batch"] = sa.Batch(ctx, [s["mesh"]] * count)
        s["batch"].set_problem([d["k"] + case["dk"] * f for f in range(count)], [d["dirs"]] * count)
        s["net"] = warmstart.WarmStartMLP(ctx, case["width"], seed=3)
        s["net"].set_params(_he_parameters(d["rng"], case["width"]))
        s["net"].set_dataset(*_samples(d["rng"], 50000))
        s["net"].train(100, batch=4096)
        return s
    s["workspace"] = sa.TbemAssemblyWorkspace(ctx, s["mesh"])
    s["system"] = sa.TbemSystem(ctx, n)
    s["incident"] = sa.IncidentField(d["dirs"])
    if kind == "solve":
        s["operator"] = sa.DenseMatrixOperator(s["system"])
    elif kind == "assemble":
        s["views"] = _system_views(s["system"])
    elif kind == "derivative":
        s["slope"] = sa.TbemSystem(ctx, n)
        s["views"] = _system_views(s["system"]) + _system_views(s["slope"])
    else:
        cols = case.get("columns", 1)
        s["X"] = sa.DeviceVector(ctx, n * cols)
        s["out"] = _view(s["X"], s["X"].ptr, (n, cols))
        s["operator"] = sa.DenseMatrixOperator(s["system"])
        if kind == "refine":
            s["B"] = sa.DeviceVector(ctx, n * cols)
            s["copy"] = sa.LowpMatrix(s["system"], case["format"])
        else:
            s["workspace"].assemble(physics, s["beta"], s["system"])
            if kind == "product":
                s["B"] = _device_block(d["X"])
            else:
                s["B"] = sa.DeviceVector(ctx, n * cols)
                s["incident"].write_device(s["B"], s["mesh"], physics, s["beta"])
    ctx.synchronize()
    return s


# --------------------------------------------------------------------------
# One pass


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "train":
        net = warmstart.WarmStartMLP(context(), case["width"], seed=3)
        net.set_params(s["parameters"])
        net.set_dataset(s["raw"], s["targets"])
        losses = net.train(case["steps"], batch=case["batch"], seed=5)
        p = net.params()
        net.close()
        return {"losses": losses, "parameters": p}
    if kind == "field":
        f = sa.compute_total_field(s["points"], s["mesh"], s["p"], s["wave"], s["physics"], s["v"])
        return {"scattered": f.p_scattered, "total": f.p_total}
    if kind in ("batch", "sweep"):
        b = s["batch"]
        b.assemble()
        fmt = case.get("format", "fp16_ir")
        if fmt != "fp64":
            b.convert(fmt[:4])
        if kind == "sweep":
            b.learned_guesses(s["net"])
        b.solve(fmt, restart=50 if fmt == "fp64" else 30, max_cycles=30, tolerance=1e-8, inner_tolerance=1e-3,
                use_guess=kind == "sweep")
        return np.concatenate([x.reshape(-1) for x in b.solutions()])
    physics, beta, system, mesh = s["physics"], s["beta"], s["system"], s["mesh"]
    if kind == "solve":
        s["workspace"].assemble(physics, beta, system)
        s["incident"].add_to_system(system, mesh, physics, beta)
        config = sa.GmresConfig(max_iterations=20, restart=case["restart"], tolerance=1e-8)
        return sa.gmres(s["operator"], system.rhs, config).x
    if kind == "assemble":
        s["workspace"].assemble(physics, beta, system)
        s["incident"].add_to_system(system, mesh, physics, beta)
        return {"matrix": s["views"][0], "rhs": s["views"][1]}
    if kind == "derivative":
        s["workspace"].assemble(physics, beta, system)
        s["workspace"].assemble_wavenumber_derivative(physics, system=s["slope"])
        a, b, da, db = s["views"]
        return {"matrix": a, "rhs": b, "matrix_slope": da, "rhs_slope": db}
    if kind == "gmres":
        config = sa.GmresConfig(max_iterations=20, restart=case["restart"], tolerance=1e-8)
        sa.gmres_device(s["operator"], s["B"].ptr, s["X"], config)
    elif kind == "product":
        s["operator"].apply_block_device(s["B"], s["X"], case["columns"])
    elif kind == "solve_many":
        config = sa.BlockGmresConfig(max_iterations=20, restart=case["restart"], tolerance=1e-8)
        sa.block_gmres_device(s["operator"], s["B"], case["columns"], s["X"], config)
    else:
        s["workspace"].assemble(physics, beta, system)
        s["incident"].write_device(s["B"], mesh, physics, beta)
        s["copy"].update()
        config = sa.GmresIrConfig(max_outer_iterations=20, outer_tolerance=1e-8, max_inner_iterations=50)
        sa.gmres_ir_device(s["operator"], s["copy"], s["B"], case["columns"], s["X"], config)
    return s["out"]


# --------------------------------------------------------------------------
# What a pass cannot do without

EVALUATION = 70.0  # FP64 operations of one kernel evaluation (square root, division, sincos counted once each)
PRODUCTS = 40.0    # Krylov products of a solve to 1e-8 at a resolved wavenumber


def _assembly_work(n):
    return {"bytes": 16.0 * n * n, "flops": 13.0 * EVALUATION * n * n}


def work(case):
    kind = case["kind"]
    if kind == "train":
        w, m, t = case["width"], float(case["batch"]), float(case["steps"])
        weights = 64.0 * w + 2.0 * w * w + 2.0 * w
        # every layer's products three times (forward, input gradient, weight gradient)
        return {"bytes": t * (48.0 * m + 28.0 * weights), "flops": t * 6.0 * m * weights}
    if kind == "batch":
        bytes_, flops = 0.0, 0.0
        for i in range(case["instances"]):
            n, c = 20.0 * 4 ** (2 + i % (case["level_max"] - 1)), 1 + (5 * i + 3) % 16
            a = _assembly_work(n)
            half = 1.0 if case["format"] == "fp64" else 0.25
            # the matrix written, read for the copy and for the products of the solve
            bytes_ += a["bytes"] * (1 + PRODUCTS * half)
            flops += a["flops"] + PRODUCTS * 8.0 * n * n * c
        return {"bytes": bytes_, "flops": flops}
    n = float(_panels(case))
    a = _assembly_work(n)
    cols = float(case.get("columns", 1))
    if kind == "field":
        return {"bytes": 112.0 * n + 72.0 * case["points"], "flops": 7.0 * 47.0 * n * case["points"]}
    if kind == "sweep":
        f = float(case["instances"])
        # one evaluation of the geometry per point for all members, about 20 operations per member
        return {"bytes": f * a["bytes"] * (1 + 0.25 * PRODUCTS),
                "flops": n * n * 13.0 * (EVALUATION + 20.0 * f) + f * PRODUCTS * 8.0 * n * n}
    if kind == "solve":
        return {"bytes": a["bytes"], "flops": a["flops"] + PRODUCTS / 2 * 8.0 * n * n}
    if kind == "assemble":
        return a
    if kind == "derivative":
        return {"bytes": 2 * a["bytes"], "flops": 2.5 * a["flops"]}
    if kind == "product":
        return {"bytes": a["bytes"] + 32.0 * n * cols, "flops": 8.0 * n * n * cols}
    if kind == "gmres":
        return {"bytes": PRODUCTS * 16.0 * n * n, "flops": PRODUCTS * 8.0 * n * n}
    if kind == "solve_many":
        return {"bytes": 0.75 * PRODUCTS * 16.0 * n * n, "flops": 0.75 * PRODUCTS * 8.0 * n * n * cols}
    # refinement: assembly, the copy, about PRODUCTS low-precision and 4 FP64 products
    return {"bytes": (1 + 1 + 0.25 + 0.25 * PRODUCTS + 4) * 16.0 * n * n,
            "flops": a["flops"] + (PRODUCTS + 4) * 8.0 * n * n * cols}


def tolerance(case):
    """About four times what two correct evaluations differ by (measured against ``exact``)."""
    kind = case["kind"]
    if kind == "field":
        return {"rel": 1e-14}
    if kind in ("assemble", "product"):
        return {"rel": 2e-13}  # the rounding of points on nearly touching panels, relative to the panel size
    if kind == "derivative":
        return {"rel": 4e-13}
    if kind == "train":
        return {"rel": 8e-3}  # BF16 layers; a rounding travels through every later step
    return {"rel": 4e-8}  # solved to a relative residual of 1e-8


# --------------------------------------------------------------------------
# The same results in plain FP64 torch

TR13 = (  # (s, t, weight) of the 13-point triangle rule
    [(0.333333333333333, 0.333333333333333, -0.149570044467682)]
    + [(s, t, 0.175615257433208) for s, t in ((0.260345966079040, 0.260345966079040),
                                               (0.260345966079040, 0.479308067841920),
                                               (0.479308067841920, 0.260345966079040))]
    + [(s, t, 0.053347235608838) for s, t in ((0.065130102902216, 0.065130102902216),
                                               (0.065130102902216, 0.869739794195568),
                                               (0.869739794195568, 0.065130102902216))]
    + [(s, t, 0.077113760890257) for a, b, c in ((0.048690315425316, 0.312865496004874, 0.638444188569810),)
       for s, t in ((a, b), (b, a), (a, c), (c, a), (b, c), (c, b))])
TR7 = ([(0.333333333333333, 0.333333333333333, 0.225)]
       + [(s, t, 0.125939180544827) for s, t in ((0.797426985353087, 0.101286507323456),
                                                  (0.101286507323456, 0.797426985353087),
                                                  (0.101286507323456, 0.101286507323456))]
       + [(s, t, 0.132394152788506) for s, t in ((0.470142064105115, 0.059715871789770),
                                                  (0.059715871789770, 0.470142064105115),
                                                  (0.470142064105115, 0.470142064105115))])


class _Reference:
    """The assembled system of one mesh and wavenumber, with its wavenumber derivative if asked."""

    def __init__(self, mesh, k, bc_type=None, bc_value=None, admittance=None, slope=False):
        dev = torch.device("cuda")
        f = lambda a, t=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=t, device=dev)  # noqa: E731
        self.k, self.slope, self.dev = k, slope, dev
        v = f(mesh.nodes[mesh.triangles])
        self.v = v
        self.e1, self.e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
        cr = torch.linalg.cross(self.e1, self.e2)
        self.jac = cr.square().sum(1).sqrt()
        self.nf = cr / self.jac[:, None]
        self.area = self.jac / 2
        self.c = ((v[:, 0] + v[:, 1]) + v[:, 2]) / 3  # the rounded collocation point is data to both sides
        out = torch.sign((self.nf * self.c).sum(1))
        self.nx = self.nf * torch.where(out < 0, -1.0, 1.0)[:, None]
        n = self.n = v.shape[0]
        self.pressure = f(bc_type) == 1 if bc_type is not None else torch.zeros(n, dtype=torch.bool, device=dev)
        z = torch.zeros(n, dtype=torch.complex128, device=dev)
        self.adm = z if admittance is None else f(np.nan_to_num(admittance), torch.complex128)
        self.value = z if bc_value is None else f(bc_value, torch.complex128)
        self.general = bc_type is not None
        self.beta, self.dbeta = 1j / k, -1j / k ** 2
        self.iwr, self.diwr = 1j * 1.21 * 343.0 * k, 1j * 1.21 * 343.0

    def channels(self, diff, nx, nf, w):
        """G, H, Ht, E of a quadrature point at diff = y - x with weight w, and their k derivatives."""
        k = self.k
        r = diff.square().sum(-1).sqrt()
        inv = 1 / r
        pn, qn = (diff * nf).sum(-1) * inv, -(diff * nx).sum(-1) * inv
        nn, rq = (nx * nf).sum(-1), pn * qn
        g = torch.polar(w * inv / (4 * math.pi), k * r)
        z1 = torch.complex(-inv, torch.full_like(inv, k))
        t3 = 3 * rq + nn
        ef = torch.complex((3 * inv * inv - k * k) * rq + nn * inv * inv, -k * inv * t3)
        b = g * z1
        val = (g, b * pn, b * qn, g * ef)
        if not self.slope:
            return val, None
        dg = 1j * r * g
        db = dg * z1 + 1j * g
        return val, (dg, db * pn, db * qn, dg * ef + g * torch.complex(-2 * k * rq, -inv * t3))

    def entry(self, ch, dch, j):
        """Matrix coefficient (and derivative) of columns j from their channel sums; and the right-hand-side part."""
        g, h, ht, e = ch
        cb, hb = h + self.beta * e, g + self.beta * ht
        p, y = self.pressure[j], self.adm[j]
        a = torch.where(p, -hb, cb - self.iwr * y * hb)
        val = self.value[j]
        rhs = torch.where(p, val * cb, val * self.iwr * hb)
        if dch is None:
            return a, rhs, None, None
        dg, dh, dht, de = dch
        dcb = dh + self.beta * de + self.dbeta * e
        dhb = dg + self.beta * dht + self.dbeta * ht
        da = torch.where(p, -dhb, dcb - y * (self.iwr * dhb + self.diwr * hb))
        drhs = torch.where(p, val * dcb, val * (self.iwr * dhb + self.diwr * hb))
        return a, rhs, da, drhs

    def assemble(self):
        n, dev = self.n, self.dev
        out = [torch.empty((n, n), dtype=torch.complex128, device=dev) for _ in range(2 if self.slope else 1)]
        near = []
        rhs = [torch.zeros(n, dtype=torch.complex128, device=dev) for _ in out]
        driven = torch.nonzero(self.value != 0).reshape(-1)
        step = max(1, 6000000 // n)
        jj = torch.arange(n, device=dev)
        root = self.area.sqrt()
        for i0 in range(0, n, step):
            i = torch.arange(i0, min(n, i0 + step), device=dev)
            x, nx = self.c[i][:, None], self.nx[i][:, None]
            dist = (self.c[None] - x).square().sum(-1).sqrt()
            hit = dist / root[None] < 3.0
            hit[torch.arange(i.numel(), device=dev), i] = False
            at = torch.nonzero(hit)
            near.append(torch.stack([at[:, 0] + i0, at[:, 1]], 1))
            ch = dch = None
            for s, t, w in TR13:
                diff = (self.v[:, 0][None] - x) + (s * self.e1 + t * self.e2)[None]
                diff = torch.where(diff.square().sum(-1, keepdim=True) > 1e-28, diff, 1.0)  # the diagonal comes later
                c, d = self.channels(diff, nx, self.nf[None], 0.5 * w * self.jac[None])
                ch = c if ch is None else tuple(p + q for p, q in zip(ch, c))
                if d is not None:
                    dch = d if dch is None else tuple(p + q for p, q in zip(dch, d))
            self._put(out, rhs, driven, i[:, None].expand(-1, n), jj[None].expand(i.numel(), -1), ch, dch, rows=i,
                      skip=hit)
        near = torch.cat(near)
        for p0 in range(0, near.shape[0], 100000):
            self._near(out, rhs, near[p0:p0 + 100000])
        self._self(out, rhs)
        return out, rhs

    def _put(self, out, rhs, driven, i, j, ch, dch, rows=None, skip=None):
        a, b, da, db = self.entry(ch, dch, j)
        for m, v in zip(out, (a, da)):
            if rows is not None:
                m[rows] = v
            else:
                m[i, j] = v
        if driven.numel():
            for r, v in zip(rhs, (b, db)):
                if rows is not None:
                    v = torch.where(skip | (i == j), 0.0, v)
                    r[rows] += v.sum(1)
                else:
                    r.index_add_(0, i, v)

    def _near(self, out, rhs, pairs):
        """Subdivided pairs: cells nearer than 3 of their size are quartered, level by level; a level stops at
        its 16th such cell, and at most 110 cells are kept."""
        dev = self.dev
        np_ = pairs.shape[0]
        src, v = self.c[pairs[:, 0]], self.v[pairs[:, 1]]
        area = self.area[pairs[:, 1]]
        owner = torch.arange(np_, device=dev)
        cells = torch.tensor([[0.0, 0.0], [1.0, 0.0], [0.0, 1.0]], dtype=torch.float64, device=dev).expand(np_, 3, 2)
        kept = torch.zeros(np_, dtype=torch.int64, device=dev)
        ch = [torch.zeros(np_, dtype=torch.complex128, device=dev) for _ in range(8)]
        scale = 1.0
        while owner.numel():
            mid = cells.sum(1) / 3
            e1, e2 = v[owner, 1] - v[owner, 0], v[owner, 2] - v[owner, 0]
            pos = v[owner, 0] + mid[:, :1] * e1 + mid[:, 1:] * e2
            ratio = (pos - src[owner]).square().sum(1).sqrt() / (area[owner].sqrt() * scale)
            split = ratio < 3.0
            first = torch.searchsorted(owner, owner)  # owners are sorted
            run = torch.cumsum(split.long(), 0)
            before = run - split.long()
            seen = run - before[first]
            leaf = ~split & (seen <= 15)
            lrun = torch.cumsum(leaf.long(), 0)
            rank = lrun - leaf.long() - (lrun - leaf.long())[first] + kept[owner]
            use = leaf & (rank < 110)
            kept.index_add_(0, owner[leaf], torch.ones_like(owner[leaf]))
            self._leaves(ch, owner[use], cells[use], pairs)
            grow = split & (seen <= 15)
            o, q = owner[grow], cells[grow]
            m01, m12, m20 = (q[:, 0] + q[:, 1]) / 2, (q[:, 1] + q[:, 2]) / 2, (q[:, 2] + q[:, 0]) / 2
            kids = torch.stack([torch.stack([q[:, 0], m01, m20], 1), torch.stack([q[:, 1], m12, m01], 1),
                                torch.stack([q[:, 2], m20, m12], 1), torch.stack([m01, m12, m20], 1)], 1)
            cells = kids.reshape(-1, 3, 2)
            owner = o.repeat_interleave(4)
            scale *= 0.5
        driven = torch.nonzero(self.value != 0).reshape(-1)
        self._put(out, rhs, driven, pairs[:, 0], pairs[:, 1], ch[:4], ch[4:] if self.slope else None)

    def _leaves(self, ch, owner, cells, pairs):
        i, j = pairs[owner, 0], pairs[owner, 1]
        a, b = cells[:, 1] - cells[:, 0], cells[:, 2] - cells[:, 0]
        det = (a[:, 0] * b[:, 1] - b[:, 0] * a[:, 1]).abs()
        for s, t, w in TR13:
            local = cells[:, 0] + s * a + t * b
            diff = (self.v[j, 0] - self.c[i]) + (local[:, :1] * self.e1[j] + local[:, 1:] * self.e2[j])
            c, d = self.channels(diff, self.nx[i], self.nf[j], 0.5 * w * det * self.jac[j])
            for q, val in enumerate(c + (d or ())):
                ch[q].index_add_(0, owner, val)

    def _self(self, out, rhs):
        """Self panels: edge integral of the hypersingular part and collapsed Gauss rules of the weakly singular ones."""
        dev, k = self.dev, self.k
        ka = k * self.area.sqrt().clamp_min(1e-10)
        beta, iwr = self.beta, self.iwr
        for lo, hi, ngp, ng, nsec1, nsec2 in ((0, 0.3, 3, 4, 4, 2), (0.3, 1, 4, 5, 6, 2), (1, 2, 5, 6, 8, 3),
                                              (2, math.inf, 6, 7, 10, 4)):
            j = torch.nonzero((ka >= lo) & (ka < hi)).reshape(-1)
            if not j.numel():
                continue
            x, nx, nf, v, jac = self.c[j], self.nx[j], self.nf[j], self.v[j], self.jac[j]
            ch = [torch.zeros(j.numel(), dtype=torch.complex128, device=dev) for _ in range(8)]
            gx, gw = np.polynomial.legendre.leggauss(ngp)
            for e in range(3):
                edge = v[:, (e + 1) % 3] - v[:, e]
                length = edge.square().sum(1).sqrt()
                unit = edge / length[:, None]
                for sec in range(nsec1):
                    mid = -1.0 - 1.0 / nsec1 + (sec + 1) * 2.0 / nsec1
                    for g0, w0 in zip(gx, gw):
                        diff = (v[:, e] - x) + edge * ((mid + g0 / nsec1 + 1.0) / 2)
                        r = diff.square().sum(1).sqrt()
                        g = torch.polar(w0 * length / (2 * nsec1) / (4 * math.pi * r), k * r)
                        z1 = torch.complex(-1 / r, torch.full_like(r, k))
                        turn = (torch.linalg.cross(diff / r[:, None], unit) * nx).sum(1)
                        ch[3] += g * z1 * turn
                        ch[7] += (1j * r * g * z1 + 1j * g) * turn
            gx, gw = np.polynomial.legendre.leggauss(ng)
            csi, eta = (0.0, 1.0, 0.0, 0.5, 0.5, 0.0), (0.0, 0.0, 1.0, 0.0, 0.5, 0.5)
            nn = (nx * nf).sum(1)
            for e in range(3):
                for sec in range(nsec2):
                    p, q = (e, e + 3) if sec == 0 else (e + 3, (e + 1) % 3)
                    for a0, wa in zip(gx, gw):
                        for b0, wb in zip(gx, gw):
                            s = 0.5 * (1 - a0) / 3 + 0.25 * (1 + a0) * ((1 - b0) * csi[p] + (1 + b0) * csi[q])
                            t = 0.5 * (1 - a0) / 3 + 0.25 * (1 + a0) * ((1 - b0) * eta[p] + (1 + b0) * eta[q])
                            diff = (v[:, 0] - x) + (s * self.e1[j] + t * self.e2[j])
                            r = diff.square().sum(1).sqrt()
                            g = torch.polar(wa * wb * (1 + a0) / (24.0 * nsec2) * jac / (4 * math.pi * r), k * r)
                            z1 = torch.complex(-1 / r, torch.full_like(r, k))
                            dg = 1j * r * g
                            b, db = g * z1, dg * z1 + 1j * g
                            pn, qn = (diff * nf).sum(1) / r, -(diff * nx).sum(1) / r
                            for m, val in enumerate((g, b * pn, b * qn, k * k * nn * g, dg, db * pn, db * qn,
                                                     nn * (k * k * dg + 2 * k * g))):
                                ch[m] += val
            a, b, da, db = self.entry(ch[:4], ch[4:] if self.slope else None, j)
            p, y, val = self.pressure[j], self.adm[j], self.value[j]
            out[0][j, j] = a + torch.where(p, 0.5 * beta, -0.5 - 0.5 * iwr * beta * y)
            rhs[0][j] += b + torch.where(p, -0.5 * val, 0.5 * iwr * beta * val)
            if self.slope:
                slope = self.diwr * beta + iwr * self.dbeta
                out[1][j, j] = da + torch.where(p, 0.5 * self.dbeta, -0.5 * slope * y)
                rhs[1][j] += db + torch.where(p, 0.0, 0.5 * slope * val)

    def waves(self, dirs):
        """Right-hand sides -(p + beta dp/dn) of unit plane waves."""
        d = torch.as_tensor(dirs, dtype=torch.float64, device=self.dev)
        d = d / d.square().sum(1, keepdim=True).sqrt()
        p = torch.polar(torch.ones((), dtype=torch.float64, device=self.dev), self.k * (self.c @ d.T))
        return -(p + self.beta * 1j * self.k * (self.nx @ d.T) * p)


def _matmul(a, x):
    """a @ x in complex128 (column by column for few columns, as plain matrix-vector products)."""
    return torch.stack([torch.mv(a, x[:, c].contiguous()) for c in range(x.shape[1])], 1) if x.shape[1] < 4 else a @ x


def _solve(a, b):
    """a x = b by GMRES on every column together, to the rounding level (two cycles)."""
    n, cols = b.shape
    m = min(70, n)
    x = torch.zeros_like(b)
    for _ in range(2):
        r = b - _matmul(a, x)
        beta = r.abs().square().sum(0).sqrt()
        basis = torch.empty((m + 1, n, cols), dtype=torch.complex128, device=b.device)
        basis[0] = r / beta
        h = torch.zeros((cols, m + 1, m), dtype=torch.complex128, device=b.device)
        for j in range(m):
            w = _matmul(a, basis[j])
            for _ in range(2):
                c = (basis[:j + 1].conj() * w[None]).sum(1)
                w = w - (basis[:j + 1] * c[:, None]).sum(0)
                h[:, :j + 1, j] += c.T
            s = w.abs().square().sum(0).sqrt()
            h[:, j + 1, j] = s
            basis[j + 1] = w / s.clamp_min(1e-300)
        hh = h.cpu().numpy()
        y = np.zeros((cols, m), dtype=np.complex128)
        for c in range(cols):
            e = np.zeros(m + 1, dtype=np.complex128)
            e[0] = float(beta[c])
            y[c] = np.linalg.lstsq(hh[c], e, rcond=1e-15)[0]
        x = x + (basis[:m] * torch.as_tensor(y.T.copy(), device=b.device)[:, None]).sum(0)
    return x


def _exact_field(case, d):
    dev = torch.device("cuda")
    ref = _Reference(d["mesh"], d["k"])
    pts = torch.as_tensor(d["points"], device=dev)
    p = torch.as_tensor(d["p"], device=dev)
    v = torch.zeros_like(p) if d["v"] is None else torch.as_tensor(d["v"], device=dev)
    out = torch.zeros(pts.shape[0], dtype=torch.complex128, device=dev)
    for i0 in range(0, pts.shape[0], 512):
        x = pts[i0:i0 + 512, None]
        for s, t, w in TR7:
            diff = (ref.v[:, 0] + s * ref.e1 + t * ref.e2)[None] - x
            r = diff.square().sum(-1).sqrt()
            g = torch.polar(0.5 * w * ref.jac[None] / (4 * math.pi * r), d["k"] * r)
            dn = (diff * ref.nf[None]).sum(-1) / r
            out[i0:i0 + 512] += (g * torch.complex(-1 / r, torch.full_like(r, d["k"])) * dn) @ p - ref.iwr * (g @ v)
    wave = d["dirs"][0] / np.linalg.norm(d["dirs"][0])
    inc = np.exp(1j * d["k"] * (d["points"] @ wave))
    out = out.cpu().numpy()
    return {"scattered": out, "total": out + inc}


def _exact_train(case, seed):
    """The training run without any rounding to BF16: features, SiLU layers, half squared error, Adam."""
    d = _inputs(case, seed)
    dev, w = torch.device("cuda"), case["width"]
    flat = _he_parameters(d["rng"], w)
    raw, targets = _samples(d["rng"], case["samples"])
    raw = torch.as_tensor(raw, device=dev).double()
    targets = torch.as_tensor(targets, device=dev).double()
    c, nn, dr, k = raw[:, 0:3], raw[:, 3:6], raw[:, 6:9], raw[:, 9:10] / 12.0
    dc, dn = (dr * c).sum(1, keepdim=True), (dr * nn).sum(1, keepdim=True)
    feats = [c, nn, dr, k, dn, dc]
    for q in (dc, dn, k, k * dc):
        for level in range(6):
            feats += [torch.sin(math.pi * 2 ** level * q), torch.cos(math.pi * 2 ** level * q)]
    feats.append(torch.zeros((raw.shape[0], 4), dtype=torch.float64, device=dev))
    feats = torch.cat(feats, 1)
    shapes = ((w, 64), (w, w), (w, w), (2, w))
    p = torch.as_tensor(flat, device=dev).double()
    m1, m2 = torch.zeros_like(p), torch.zeros_like(p)
    losses = []
    count, batch = case["samples"], case["batch"]
    for step in range(case["steps"]):
        with np.errstate(over="ignore"):
            start = np.uint64((5 * 0x100000001B3 + step) & 0xFFFFFFFFFFFFFFFF)
            z = start + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, batch + 1, dtype=np.uint64)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z ^= z >> np.uint64(31)
        at = torch.as_tensor((z % np.uint64(count)).astype(np.int64), device=dev)
        q = p.clone().requires_grad_(True)
        a, o = feats[at], 0
        for layer, (rows, cols) in enumerate(shapes):
            weight, bias = q[o:o + rows * cols].view(rows, cols), q[o + rows * cols:o + rows * cols + rows]
            o += rows * cols + rows
            a = a @ weight.T + bias
            if layer < 3:
                a = a * torch.sigmoid(a)
        loss = (a - targets[at]).square().sum() / (2 * batch)
        loss.backward()
        g = q.grad
        frac = step / (case["steps"] - 1) if case["steps"] > 1 else 0.0
        lr = 5e-5 + 0.5 * (2e-3 - 5e-5) * (1 + math.cos(math.pi * frac))
        m1 = 0.9 * m1 + 0.1 * g
        m2 = 0.999 * m2 + 0.001 * g * g
        p = p - lr * (m1 / (1 - 0.9 ** (step + 1))) / ((m2 / (1 - 0.999 ** (step + 1))).sqrt() + 1e-8)
        losses.append(float(loss.detach()))
    return {"losses": np.array(losses), "parameters": p.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    d = _inputs(case, seed)
    if kind == "field":
        return _exact_field(case, d)
    if kind == "batch":
        if sum(m.num_elements ** 2 for m in d["meshes"]) > 4e8:
            return None  # hundreds of right-hand sides on large bodies: over 20 seconds
        parts = []
        for m, k, dirs in zip(d["meshes"], d["ks"], d["dirs"]):
            ref = _Reference(m, k)
            parts.append(_solve(ref.assemble()[0][0], ref.waves(dirs)).reshape(-1).cpu().numpy())
        return np.concatenate(parts)
    if kind == "sweep":
        parts = []
        for f in range(case["instances"]):
            ref = _Reference(d["mesh"], d["k"] + case["dk"] * f)
            parts.append(_solve(ref.assemble()[0][0], ref.waves(d["dirs"])).reshape(-1).cpu().numpy())
        return np.concatenate(parts)
    ref = _Reference(d["mesh"], d["k"], d.get("bc_type"), d.get("bc_value"), d.get("admittance"),
                     slope=kind == "derivative")
    a, rhs = ref.assemble()
    if kind == "assemble":
        return {"matrix": a[0], "rhs": rhs[0] + ref.waves(d["dirs"])[:, 0]}
    if kind == "derivative":
        return {"matrix": a[0], "rhs": rhs[0], "matrix_slope": a[1], "rhs_slope": rhs[1]}
    if kind == "product":
        return _matmul(a[0], torch.as_tensor(d["X"], device="cuda"))
    x = _solve(a[0], ref.waves(d["dirs"]))
    return x[:, 0].cpu().numpy() if kind == "solve" else x
