"""The work a user of this framework has it do, as cases that can be timed and compared.

The framework advances a NonhydrostaticModel; a program builds a model, sets its fields and then
calls ``time_step`` (once per iteration from ``Simulation``/``run``, or several steps at once
between two callbacks).  So most cases are time steps, over the configurations of the workloads,
tests and benchmark: two-dimensional turbulence, free convection (uniform and stretched z), wind
and convection with temperature and salinity, periodic DNS with the default Centered advection, the
immersed seamount with the conjugate-gradient solver, and an ensemble; FP32 and FP64; powers of two
and ragged sizes; from launch-bound grids to the largest one.  One case is the evaluation of a state
(``update_state``) by itself.

``prepare`` builds the model and its fields from the seed; ``run`` makes one pass and returns the
model's own device buffers; ``exact`` repeats the pass in plain FP64 torch, written from the
discretisation itself.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oceananigans.jl_amd"))

import oceananigans_mi355x as om  # noqa: E402

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
ENSEMBLE_SIZES = ((64, 64, 64), (96, 96, 64), (128, 128, 64), (128, 128, 128))

# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------


def _case(name, flow, nx, ny, nz, precision="fp32", call="time_step", steps=1, members=1, mix=0):
    c = dict(flow=flow, nx=nx, ny=ny, nz=nz, precision=precision, call=call, steps=steps, members=members, mix=mix)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest model anyone runs: the two-dimensional turbulence example, one step per
        # iteration of a Simulation; a step is some thirty launches over 16 thousand cells
        _case("turbulence2d_128", "turbulence", 128, 128, 1, "fp64"),
        # a small LES, as in parameter studies and in developing a setup: still launch-bound
        _case("convection_32", "convection", 32, 32, 32),
        # an LES whose sizes are what the domain asks for, with an odd number of levels
        _case("convection_150x100x75", "convection", 150, 100, 75),
        # the headline LES, a few steps between two callbacks
        _case("convection_256x256x128", "convection", 256, 256, 128, steps=4),
        # the largest: wind and convection with temperature and salinity and Smagorinsky-Lilly
        _case("wind_512x512x256", "wind", 512, 512, 256),
        # double precision, for reference solutions and for anything compared with the CPU
        _case("convection_fp64_128", "convection", 128, 128, 128, "fp64"),
        # a boundary layer resolved by a stretched z (Fourier-tridiagonal pressure solver) on a
        # grid whose sides are not powers of two
        _case("stretched_192x192x96", "stretched", 192, 192, 96),
        # flow over the immersed seamount with the conjugate-gradient pressure solver
        _case("seamount_256x256x128", "seamount", 256, 256, 128),
        # triply periodic DNS with the default advection (Centered) and constant diffusivity
        _case("dns_fp64_128", "dns", 128, 128, 128, "fp64"),
        # evaluation of a state: what set!, a restart and every substage end with
        _case("update_state_384x320x96", "convection", 384, 320, 96, call="update_state"),
        # an ensemble of members of uneven sizes advanced together
        _case("ensemble_12", "convection", 0, 0, 0, call="ensemble", steps=2, members=12, mix=5),
    ]


def draw(rng):
    def size(lo, hi):
        n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        step = rng.choice((1, 1, 2, 8, 16, 32))
        return max(lo, min(hi, int(round(n / step)) * step))

    flow = rng.choice(("turbulence", "convection", "convection", "convection", "wind", "stretched", "seamount", "dns", "ensemble"))
    precision = rng.choice(("fp32", "fp32", "fp64"))
    steps = rng.choice((1, 1, 2, 4))
    if flow == "turbulence":
        return _case(None, flow, size(64, 1024), size(64, 1024), 1, rng.choice(("fp32", "fp64")), steps=steps)
    if flow == "ensemble":
        return _case(None, "convection", 0, 0, 0, "fp32", "ensemble", rng.choice((2, 4)), rng.randrange(4, 13), rng.randrange(1, 1000))
    most = {"seamount": 1_500_000, "dns": 4_000_000}.get(flow, 6_000_000)
    while True:
        nx, ny, nz = size(24, 512), size(24, 512), size(16, 256)
        if nx * ny * nz <= most:
            break
    if flow == "seamount":
        return _case(None, flow, nx, ny, nz, "fp32")
    call = "update_state" if flow == "convection" and rng.random() < 0.2 else "time_step"
    return _case(None, flow, nx, ny, nz, precision, call, 1 if call != "time_step" else steps)


# ------------------------------------------------------------------------------------------------
# configurations and inputs
# ------------------------------------------------------------------------------------------------


def _sizes(case):
    """[(nx, ny, nz)] of the case's members."""
    if case["call"] != "ensemble":
        return [(case["nx"], case["ny"], case["nz"])]
    pick = np.random.default_rng(case["mix"])
    return [ENSEMBLE_SIZES[int(pick.integers(len(ENSEMBLE_SIZES)))] for _ in range(case["members"])]


def _faces(nz, depth, ratio):
    """Geometrically stretched z faces, finest at the surface."""
    d = depth * (ratio - 1) / (ratio ** nz - 1) * ratio ** np.arange(nz)
    f = -np.concatenate([[0.0], np.cumsum(d)])[::-1]
    f[0], f[-1] = -depth, 0.0
    return f


def _hill(x, y, side, depth):
    return -depth + 0.6 * depth * np.exp(-((x - side / 2) ** 2 + (y - side / 2) ** 2) / (0.15 * side) ** 2)


def _setup(flow, n):
    """The flow on a grid of size n, in plain numbers: domain, physics, time step."""
    nx, ny, nz = n
    # u0: velocity scale (a time step carries the flow a tenth of a cell or so), n2 and db: background
    # stratification and buoyancy (or temperature) noise
    s = dict(n=n, periodic_z=False, flat=False, faces=None, bottom=None, weno=True, closure=None, f=0.0, tracers=(), buoyancy=None,
             flux={}, gradient={}, u0=0.1, mean_u=0.0, solver=None)
    if flow == "turbulence":
        return dict(s, L=(2 * np.pi, 2 * np.pi, 1.0), flat=True, u0=0.5, dt=0.1 * 2 * np.pi / max(nx, ny))
    if flow == "dns":
        return dict(s, L=(2 * np.pi,) * 3, periodic_z=True, weno=False, closure=("constant", 5e-3, 5e-3), tracers=("c",), u0=0.5,
                    dt=0.1 * 2 * np.pi / max(n))
    if flow == "convection":
        return dict(s, L=tuple(map(float, n)), closure=("amd", 1 / 3, 1 / 3), f=1e-4, tracers=("b",), buoyancy="b", flux={"b": (None, 1e-8)},
                    n2=1e-6, db=1e-5, dt=1.0)
    if flow == "stretched":
        return dict(s, L=(float(nx), float(ny), float(nz)), faces=_faces(nz, float(nz), 1 + 2 / nz), closure=("amd", 1 / 3, 1 / 3), f=1e-4,
                    tracers=("b",), buoyancy="b", n2=1e-6, db=1e-5, dt=0.5, mean_u=0.1)
    if flow == "wind":
        return dict(s, L=tuple(map(float, n)), closure=("smagorinsky", 0.16, 1.0, 1.0), tracers=("T", "S"), buoyancy="TS",
                    flux={"u": (None, -1e-4), "T": (None, 200.0 / (1026.0 * 3991.0))}, gradient={"T": (0.01, None)}, n2=0.01, db=1e-3, dt=1.0)
    if flow == "seamount":
        side, depth = 10e3, 1e3
        x, y = (np.arange(nx) + 0.5) * side / nx, (np.arange(ny) + 0.5) * side / ny
        return dict(s, L=(side, side, depth), faces=_faces(nz, depth, 1.02), bottom=_hill(x[:, None], y[None, :], side, depth),
                    closure=("amd", 1 / 3, 1 / 3), tracers=("b",), buoyancy="b", n2=1e-6, db=1e-7, dt=4.0, u0=1e-2, mean_u=0.1,
                    solver="cg")
    raise ValueError(flow)


ALPHA, BETA, GRAVITY = 2e-4, 8e-4, 9.80665


def _model(s, precision):
    ft = np.float32 if precision == "fp32" else np.float64
    (nx, ny, nz), L = s["n"], s["L"]
    if s["flat"]:
        grid = om.RectilinearGrid(float_type=ft, size=(nx, ny), x=(0, L[0]), y=(0, L[1]), topology=(om.Periodic, om.Periodic, om.Flat))
    else:
        grid = om.RectilinearGrid(float_type=ft, size=(nx, ny, nz), x=(0, L[0]), y=(0, L[1]),
                                  z=s["faces"] if s["faces"] is not None else (-L[2], 0),
                                  topology=(om.Periodic, om.Periodic, om.Periodic if s["periodic_z"] else om.Bounded))
    if s["bottom"] is not None:
        grid = om.ImmersedBoundaryGrid(grid, om.GridFittedBottom(s["bottom"]))
    kw = dict(tracers=s["tracers"], advection=om.WENO() if s["weno"] else None)
    if s["closure"]:
        kind, a = s["closure"][0], s["closure"][1:]
        kw["closure"] = {"amd": lambda: om.AnisotropicMinimumDissipation(Cnu=a[0], Ckappa=a[1]), "constant": lambda: om.ScalarDiffusivity(nu=a[0], kappa=a[1]),
                         "smagorinsky": lambda: om.SmagorinskyLilly(C=a[0], Cb=a[1], Pr=a[2])}[kind]()
    if s["buoyancy"] == "b":
        kw["buoyancy"] = om.BuoyancyTracer()
    elif s["buoyancy"] == "TS":
        kw["buoyancy"] = om.SeawaterBuoyancy(equation_of_state=om.LinearEquationOfState(ALPHA, BETA))
    if s["f"]:
        kw["coriolis"] = om.FPlane(f=s["f"])
    if s["solver"] == "cg":
        kw["pressure_solver"] = om.ConjugateGradientPoissonSolver(reltol=1e-8, abstol=0, maxiter=1000)
    bcs = {}
    for f in set(s["flux"]) | set(s["gradient"]):
        side = [None if v is None else om.FluxBoundaryCondition(v) for v in s["flux"].get(f, (None, None))]
        for q, v in enumerate(s["gradient"].get(f, (None, None))):
            if v is not None:
                side[q] = om.GradientBoundaryCondition(v)
        bcs[f] = om.FieldBoundaryConditions(bottom=side[0], top=side[1])
    if bcs:
        kw["boundary_conditions"] = bcs
    return om.NonhydrostaticModel(grid, **kw)


def _noise(gen, shape):
    """Unit-variance random field with grid-scale and larger scales, as a resolved turbulent flow has."""
    w = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float64)
    s = w
    for _ in range(3):
        for d in range(3):
            if shape[d] > 1:
                s = 0.5 * s + 0.25 * (torch.roll(s, 1, d) + torch.roll(s, -1, d))
    return 0.2 * w + s / s.std()


def _inputs(s, precision, seed, member=0):
    """{field: tensor (z, y, x) of the interior}, in the model's precision.  The velocity is the curl of
    a potential on the cell edges (zero on the walls), so it has no divergence."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(1000003 * int(seed) + member)
    nx, ny, nz = s["n"]
    walls = not (s["flat"] or s["periodic_z"])
    faces = s["faces"] if s["faces"] is not None else np.linspace(-s["L"][2], 0.0, nz + 1)
    dz = torch.as_tensor(np.diff(faces), device=DEVICE)[:, None, None]
    ddx = lambda a: (torch.roll(a, -1, 2) - a) * (nx / s["L"][0])  # noqa: E731
    ddy = lambda a: (torch.roll(a, -1, 1) - a) * (ny / s["L"][1])  # noqa: E731
    ddz = lambda a: ((a[1:] - a[:-1]) if walls else (torch.roll(a, -1, 0) - a)) / dz  # noqa: E731
    az = _noise(gen, (nz, ny, nx))
    out = {"u": ddy(az), "v": -ddx(az), "w": torch.zeros_like(az)}
    if not s["flat"]:
        ax, ay = _noise(gen, (nz, ny, nx)), _noise(gen, (nz, ny, nx))
        if walls:
            ax, ay = (torch.cat([torch.zeros_like(a[:1]), a[1:], torch.zeros_like(a[:1])]) for a in (ax, ay))
        # potentials in proportion to the spacing, so that the flow is as steep as the grid is flat
        ax, ay = (a * float(dz.mean()) * ny / s["L"][1] for a in (ax, ay))
        out = {"u": out["u"] - ddz(ay), "v": out["v"] + ddz(ax), "w": ddx(ay) - ddy(ax)}
    scale = s["u0"] / out["u"].std()
    out = {c: a * scale for c, a in out.items()}
    out["u"] += s["mean_u"]
    if s["tracers"]:
        z = torch.as_tensor(0.5 * (faces[1:] + faces[:-1]), device=DEVICE)[:, None, None]
        for c in s["tracers"]:
            n = _noise(gen, (nz, ny, nx))
            out[c] = {"b": lambda: s["n2"] * z + s["db"] * n, "T": lambda: 20 + s["n2"] * z + s["db"] * n,
                      "S": lambda: 35 + s["db"] * n, "c": lambda: n}[c]()
    t = torch.float32 if precision == "fp32" else torch.float64
    return {k: v.to(t) for k, v in out.items()}


class _Buffer:
    """A field's device memory, as om_field_info describes it; keeps its model alive."""

    def __init__(self, field):
        info, grid = field.info(), field.model.grid
        self.model = field.model
        e = info.element_size
        first = sum(h * st for h, st in zip(grid.H, info.stride)) * e
        shape = tuple(info.parent_size[d] - 2 * grid.H[d] for d in (2, 1, 0))
        self.__cuda_array_interface__ = dict(shape=shape, strides=tuple(info.stride[d] * e for d in (2, 1, 0)), typestr="<f%d" % e,
                                             data=(info.data + first, False), version=2)


def _view(field):
    return torch.as_tensor(_Buffer(field), device=DEVICE)


def _prognostic(model):
    return {**{c: model.velocities[c] for c in ("u", "v", "w")}, **{c: model.tracers[c] for c in model.tracer_names}}


def prepare(case, seed):
    flow = case["flow"]
    models, outputs = [], []
    for m, n in enumerate(_sizes(case)):
        s = _setup(flow, n)
        model = _model(s, case["precision"])
        fields = {c: _view(f) for c, f in _prognostic(model).items()}
        for c, v in _inputs(s, case["precision"], seed, m).items():
            fields[c].copy_(v)
        if DEVICE == "cuda":
            torch.cuda.synchronize()   # the model works on a stream of its own
        # set!: halos and state; the projection only where the flow is not free of divergence already
        model.fill_halo_regions()
        model.update_state()
        if s["bottom"] is not None:
            model.compute_pressure_correction(1.0)
            model.update_state()
        if case["call"] == "update_state":
            # w's tendency at the bottom wall is never used; its levels above it are
            out = {"G" + c: _view(f)[1 if c == "w" and not s["periodic_z"] else 0:n[2]] for c, f in model.Gn.items()}
            out["nu"] = _view(model.closure_fields["nu"])
            if s["closure"][0] == "amd":
                out.update({"kappa_" + c: _view(model.closure_fields["kappa_" + c]) for c in s["tracers"]})
        else:
            # over an immersed bottom the solver leaves p with a constant of no meaning
            with_p = case["call"] == "time_step" and s["bottom"] is None
            out = dict(fields, p=_view(model.pressures["pNHS"])) if with_p else fields
        models.append(model)
        outputs.append(out)
    state = dict(call=case["call"], dt=_setup(flow, _sizes(case)[0])["dt"], steps=case["steps"], models=models, outputs=outputs)
    if case["call"] == "ensemble":
        state["ensemble"] = om.Ensemble(models)
    return state


def run(state):
    if state["call"] == "ensemble":
        state["ensemble"].time_step(state["dt"], state["steps"], mode="batched")
        return state["outputs"]
    if state["call"] == "update_state":
        state["models"][0].update_state()
    else:
        state["models"][0].time_step(state["dt"], state["steps"])
    return state["outputs"][0]


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------


def work(case):
    """A step is three substages, and the pressure solve of each couples every cell, so a substage
    reads and writes its fields once in each of: tendencies (n fields in, n out), RK update (3n or 4n),
    pressure solve (source, half spectrum there and back along each axis, pressure: 10 words),
    correction (7 words): 17n + 54 words a cell and step, with n prognostic fields; CG adds its
    iterations (at least 5 FP64 vectors each; 8 iterations a solve).  Flops: a WENO reconstruction is
    about 60, a cell's closure about 200, the transforms 5 log2 N a line and axis."""
    word = 4 if case["precision"] == "fp32" else 8
    total = dict(bytes=0.0, flops=0.0)
    for nx, ny, nz in _sizes(case):
        s = _setup(case["flow"], (nx, ny, nz))
        dims = 2 if s["flat"] else 3
        n = dims + len(s["tracers"])
        cells = nx * ny * nz
        tend = dims * n * ((65 if s["weno"] else 8) + (15 if s["closure"] else 0))
        closure = 200 if s["closure"] and s["closure"][0] != "constant" else 0
        if case["call"] == "update_state":
            total["bytes"] += cells * word * (2 * n + 1 + len(s["tracers"]))
            total["flops"] += cells * (tend + closure)
            continue
        solve = 10 * word + (8 * 40 if s["solver"] == "cg" else 0)
        total["bytes"] += case["steps"] * cells * (word * (2 * n * 3 + 11 * n + 24) + 3 * solve)
        fft = 5 * (math.log2(nx) + math.log2(ny) + math.log2(max(nz, 2)))
        total["flops"] += case["steps"] * 3 * cells * (tend + closure + fft * (8 if s["solver"] == "cg" else 1) + 8 * n + 20)
    return total


# ------------------------------------------------------------------------------------------------
# the same pass in FP64 torch
# ------------------------------------------------------------------------------------------------
X, Y, Z = 2, 1, 0   # tensor axes


class _Flow:
    """The model's discretisation on whole arrays (z, y, x): finite volumes on a staggered C grid.

    Shifts wrap, which is right for the periodic axes; a Bounded z has `h` halo planes below and
    above (and one more), and what wraps into them is never selected, because the schemes narrow
    next to inactive cells (outside the domain, or below the immersed bottom)."""

    def __init__(self, s, fields):
        self.s = s
        nx, ny, nz = self.n = s["n"]
        self.bounded = not (s["flat"] or s["periodic_z"])
        self.h = 3 if self.bounded else 0
        self.axes = (X, Y) if s["flat"] else (X, Y, Z)
        self.cells = slice(self.h, self.h + nz)
        t = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEVICE)[:, None, None]  # noqa: E731
        if s["flat"]:
            dzc = dzf = np.ones(1)
        else:
            faces = s["faces"] if s["faces"] is not None else np.linspace(-s["L"][2], 0.0, nz + 1)
            dz = np.diff(faces)
            if self.bounded:
                dzc = np.concatenate([np.full(3, dz[0]), dz, np.full(4, dz[-1])])
                dzf = 0.5 * (dzc + np.roll(dzc, 1))
                dzf[0] = dzc[0]
            else:
                dzc = dzf = np.full(nz, s["L"][2] / nz)
        self.dzc, self.dzf = t(dzc), t(dzf)
        self.d = {X: s["L"][0] / nx, Y: s["L"][1] / ny}
        P = len(dzc)
        k = torch.arange(P, device=DEVICE) - self.h
        self.outside = ((k < 0) | (k >= nz))[:, None, None] if self.bounded else torch.zeros(P, 1, 1, dtype=torch.bool, device=DEVICE)
        self.inactive, self.immersed = self.outside, s["bottom"] is not None
        if self.immersed:
            zc = torch.full((P,), math.inf, dtype=torch.float64, device=DEVICE)
            zc[self.cells] = torch.as_tensor(0.5 * (faces[1:] + faces[:-1]), device=DEVICE)
            zc[:self.h] = -math.inf
            bottom = torch.as_tensor(np.ascontiguousarray(s["bottom"].T), device=DEVICE)
            self.inactive = self.outside | (zc[:, None, None] <= bottom[None])
        self.masks = {}
        self.f = {}
        for c, v in fields.items():
            a = torch.zeros(P, ny, nx, dtype=torch.float64, device=DEVICE)
            a[self.h:self.h + v.shape[0]] = v.double()
            self.f[c] = a
        self.p = torch.zeros(P, ny, nx, dtype=torch.float64, device=DEVICE)

    # ---- shifts, averages, masks
    def at(self, a, axis, n):
        """a at index + n along the axis."""
        return a if n == 0 or a.shape[axis] == 1 and axis != Z else torch.roll(a, -n, axis)

    def avg(self, a, axis, up):
        """mean of the two values around a face (up = 0) or a centre (up = 1)."""
        return 0.5 * (self.at(a, axis, up - 1) + self.at(a, axis, up)) if axis in self.axes else a

    def near(self, axis, centre, buffer):
        """any inactive node in the 2·buffer points around a face, or around a centre."""
        key = ("near", axis, centre, buffer)
        if key not in self.masks:
            node = self.inactive & self.at(self.inactive, axis, -1) if centre else self.inactive
            r = torch.zeros_like(node)
            for q in range(1, 2 * buffer + 1):
                r = r | self.at(node, axis, q - buffer - (0 if centre else 1))
            self.masks[key] = r
        return self.masks[key]

    def touching(self, loc, every):
        """nodes at a location (axes on faces) all (any) of whose cells are inactive by the immersed
        bottom rather than by the domain's end alone."""
        key = ("touching", loc, every)
        if key not in self.masks:
            def fold(m):
                r = m
                for axis in loc:
                    o = self.at(r, axis, -1)
                    r = r & o if every else r | o
                return r
            self.masks[key] = fold(self.inactive) & ~fold(self.outside)
        return self.masks[key]

    def flux(self, v, loc):
        """v, zero on the immersed periphery of its location."""
        return torch.where(self.touching(loc, False), 0.0, v) if self.immersed else v

    def diff(self, a, axis, up, loc):
        """difference across a face (up = 0) or a centre (up = 1) of values at location loc, zero next
        to an immersed node of that location."""
        v = self.at(a, axis, up) - self.at(a, axis, up - 1)
        if self.immersed:
            m = self.touching(loc, True)
            v = torch.where(self.at(m, axis, up) | self.at(m, axis, up - 1), 0.0, v)
        return v

    def spacing(self, axis, face):
        return (self.dzf if face else self.dzc) if axis == Z else self.d[axis]

    def grad(self, a, axis, up, loc):
        if axis not in self.axes:
            return torch.zeros_like(a)
        return self.diff(a, axis, up, loc) / self.spacing(axis, up == 0)

    def area(self, axis, zface=False):
        """face area normal to the axis (on z faces, of the z-face-centred volume)."""
        dz = self.dzf if zface else self.dzc
        return {X: self.d[Y] * dz, Y: self.d[X] * dz, Z: self.d[X] * self.d[Y]}[axis]

    # ---- reconstructions
    def centred(self, a, axis, up):
        """advecting value at a face (up = 0) or centre: fourth order, second next to a boundary."""
        if axis not in self.axes:
            return a
        v2 = self.avg(a, axis, up)
        if not self.s["weno"]:
            return v2
        v4 = (7 * (self.at(a, axis, up - 1) + self.at(a, axis, up)) - self.at(a, axis, up - 2) - self.at(a, axis, up + 1)) / 12
        return torch.where(self.near(axis, up == 1, 3), v2, v4)

    def upwind(self, a, axis, up, vel):
        """advected value: WENO(5), narrowing to WENO(3) and Centered(2); or Centered(2)."""
        if not self.s["weno"]:
            return self.avg(a, axis, up)
        left = vel > 0
        q = [self.at(a, axis, up + m) for m in range(-3, 3)]
        # mirrored so that the flow comes from t[0]; r[k]: the three points of stencil k from its upwind end
        t = [torch.where(left, q[m], q[5 - m]) for m in range(5)]
        # values relative to the middle of each stencil: the same indicators, without cancellation
        def beta(c, s):
            (x, _, z) = (s[0] - s[1], 0, s[2] - s[1])
            return c[0] * x * x + c[1] * x * z + c[2] * z * z
        s0, s1, s2 = (t[2], t[3], t[4]), (t[1], t[2], t[3]), (t[0], t[1], t[2])
        b0, b1, b2 = beta((10, 11, 4), s0), beta((4, 5, 4), s1), beta((4, 11, 10), s2)
        eps = float(np.float32(1e-8))
        tau = (b0 - b2).abs()
        a0, a1, a2 = 0.3 * (1 + (tau / (b0 + eps)) ** 2), 0.6 * (1 + (tau / (b1 + eps)) ** 2), 0.1 * (1 + (tau / (b2 + eps)) ** 2)
        v = (a0 * (2 * s0[0] + 5 * s0[1] - s0[2]) + a1 * (-s1[0] + 5 * s1[1] + 2 * s1[2]) + a2 * (2 * s2[0] - 7 * s2[1] + 11 * s2[2])) \
            / (6 * (a0 + a1 + a2))
        n3 = self.near(axis, up == 1, 3)
        if self.immersed or (axis == Z and self.bounded):
            b0, b1 = (t[2] - t[3]) ** 2, (t[1] - t[2]) ** 2
            tau = (b0 - b1).abs()
            a0, a1 = 2 / 3 * (1 + (tau / (b0 + eps)) ** 2), 1 / 3 * (1 + (tau / (b1 + eps)) ** 2)
            v3 = (a0 * 0.5 * (t[2] + t[3]) + a1 * (1.5 * t[2] - 0.5 * t[1])) / (a0 + a1)
            v = torch.where(n3, torch.where(self.near(axis, up == 1, 2), self.avg(a, axis, up), v3), v)
        return v

    # ---- state
    def fill(self):
        if not self.bounded:
            return
        h, nz = self.h, self.n[2]
        for c, a in self.f.items():
            if c == "w":
                a[h] = 0
                a[h + nz] = 0
                continue
            lo, hi = self.s["gradient"].get(c, (None, None))
            a[h - 1] = a[h] - (lo or 0.0) * self.dzf[h]
            a[h + nz] = a[h + nz - 1] + (hi or 0.0) * self.dzf[h + nz]

    def copy_halo(self, a):
        if self.bounded:
            a[self.h - 1] = a[self.h]
            a[self.h + self.n[2]] = a[self.h + self.n[2] - 1]
        return a

    def buoyancy(self, g=lambda a: a):
        """g (a linear operator) of the buoyancy."""
        if self.s["buoyancy"] == "b":
            return g(self.f["b"])
        return GRAVITY * (ALPHA * g(self.f["T"]) - BETA * g(self.f["S"]))

    def close_turbulence(self):
        kind = self.s["closure"][0] if self.s["closure"] else None
        self.nu, self.kappa = None, {}
        if kind in (None, "constant"):
            return
        u, v, w = self.f["u"], self.f["v"], self.f["w"]
        own = {X: u, Y: v, Z: w}
        diag = {a: self.grad(own[a], a, 1, (a,)) for a in (X, Y, Z)}
        # G[(i, j)]: gradient along i of velocity j at the edge between axes i and j
        G = {(i, j): self.grad(own[j], i, 0, (j,)) for i in (X, Y, Z) for j in (X, Y, Z) if i != j}
        mean = lambda a, i, j: self.avg(self.avg(a, i, 1), j, 1)  # noqa: E731  (edge to centre)
        if kind == "smagorinsky":
            C, Cb, _ = self.s["closure"][1:]
            s2 = sum(diag[a] ** 2 for a in diag)
            for i, j in ((X, Y), (X, Z), (Y, Z)):
                s2 = s2 + 2 * mean((0.5 * (G[i, j] + G[j, i])) ** 2, i, j)
            n2 = self.avg(self.buoyancy(lambda a: self.grad(a, Z, 0, ())), Z, 1).clamp(min=0)
            sig = torch.where(s2 == 0, 0.0, (1 - (Cb * n2 / s2).clamp(max=1)).sqrt())
            self.nu = self.copy_halo(sig * C ** 2 * (self.d[X] * self.d[Y] * self.dzc) ** (2 / 3) * (2 * s2).sqrt())
            return
        width = {X: 2 * self.d[X], Y: 2 * self.d[Y], Z: 2 * self.dzc}
        G = {(i, j): width[i] / width[j] * g for (i, j), g in G.items()}
        S = {(i, j): 0.5 * (G[i, j] + G[j, i]) for i, j in G}
        m = {(i, j): mean(g, i, j) for (i, j), g in G.items()}
        q = sum(diag[a] ** 2 for a in diag) + sum(mean(g * g, i, j) for (i, j), g in G.items())
        r = 0
        for i in (X, Y, Z):
            j, k = [a for a in (X, Y, Z) if a != i]
            r = r + diag[i] ** 3 + diag[j] * mean(G[i, j] ** 2, i, j) + diag[k] * mean(G[i, k] ** 2, i, k) \
                + 2 * diag[i] * (mean(G[i, j] * S[i, j], i, j) + mean(G[i, k] * S[i, k], i, k)) + 2 * m[i, j] * m[i, k] * mean(S[j, k], j, k)
        d2 = 3 / (1 / width[X] ** 2 + 1 / width[Y] ** 2 + 1 / width[Z] ** 2)
        Cnu, Ckappa = self.s["closure"][1:]
        self.nu = self.copy_halo(torch.where(q == 0, 0.0, -Cnu * d2 * r / q).clamp(min=0))
        # the reference takes the y gradient of w for the (y, z) term from the x-z edges
        m_yw = mean(width[Y] / width[Z] * self.grad(w, Y, 0, (Z,)), X, Z)
        for c in self.s["tracers"]:
            g = {a: width[a] * self.grad(self.f[c], a, 0, ()) for a in (X, Y, Z)}
            g1, g2 = {a: self.avg(g[a], a, 1) for a in g}, {a: self.avg(g[a] ** 2, a, 1) for a in g}
            sig = sum(g2.values())
            th = 0
            for i in (X, Y, Z):
                for j in (X, Y, Z):
                    th = th + (diag[i] * g2[i] if i == j else (m_yw if (i, j) == (Y, Z) else m[i, j]) * g1[i] * g1[j])
            self.kappa[c] = self.copy_halo(torch.where(sig == 0, 0.0, -Ckappa * d2 * th / sig).clamp(min=0))

    def hydrostatic(self):
        """p(k) = −Σ of the face buoyancy above; zero without a Bounded z."""
        if not (self.bounded and self.s["buoyancy"]):
            return None
        t = self.avg(self.buoyancy(), Z, 0) * self.dzf        # face k, below cell k
        p = torch.zeros_like(t)
        h, nz = self.h, self.n[2]
        p[h:h + nz] = -torch.flip(torch.cumsum(torch.flip(t[h + 1:h + nz + 1], (0,)), 0), (0,))
        return p

    def update(self):
        if self.immersed:
            for c in self.s["tracers"]:
                self.f[c] = self.flux(self.f[c], ())
        self.fill()
        self.close_turbulence()
        self.G = self.tendencies()

    def edge(self, a, i, j):
        """cell values at the location of the (i, j) stress."""
        return a if i == j else self.avg(self.avg(a, i, 0), j, 0)

    def tendencies(self):
        s, f = self.s, self.f
        vel = {X: "u", Y: "v", Z: "w"}
        pHY, out = self.hydrostatic(), {}
        closure = s["closure"][0] if s["closure"] else None
        for j in self.axes:                        # momentum along j, at the j faces
            zf = j == Z
            volume = self.d[X] * self.d[Y] * (self.dzf if zf else self.dzc)
            adv, vis = [], []
            for i in self.axes:                    # transport along i: fluxes at centres or (i, j) edges
                up = 1 if i == j else 0
                loc = () if i == j else (i, j)
                a = self.area(i) if i != Z else self.area(Z)
                ut = self.centred(a * f[vel[i]], j, up)
                F = self.flux(ut * self.upwind(f[vel[j]], i, up, ut), loc)
                adv.append(self.diff(F, i, 1 - up, loc))
                if closure:
                    strain = self.grad(f[vel[j]], i, up, (j,)) if i == j else \
                        0.5 * (self.grad(f[vel[j]], i, 0, (j,)) + self.grad(f[vel[i]], j, 0, (i,)))
                    nu = s["closure"][1] if closure == "constant" else self.edge(self.nu, i, j)
                    vis.append(self.diff(self.area(i, zf and i != Z) * self.flux(-2 * nu * strain, loc), i, 1 - up, loc))
            G = -sum(adv) / volume
            if j in (X, Y) and s["f"]:
                o = Y if j == X else X
                other = self.avg(self.avg(self.flux(f[vel[o]], (o,)), o, 1), j, 0)
                G = G + (s["f"] if j == X else -s["f"]) * other
            if j in (X, Y) and pHY is not None:
                G = G - self.diff(pHY, j, 0, ()) / self.d[j]
            if j == Z and pHY is None and s["buoyancy"]:
                G = G + self.avg(self.buoyancy(), Z, 0)
            out[vel[j]] = G - sum(vis) / volume if vis else G
        volume = self.d[X] * self.d[Y] * self.dzc
        for c in s["tracers"]:
            adv, dif = [], []
            for i in self.axes:
                F = self.area(i) * f[vel[i]] * self.upwind(f[c], i, 0, f[vel[i]])
                adv.append(self.diff(self.flux(F, (i,)), i, 1, (i,)))
                if closure:
                    kappa = s["closure"][2] if closure == "constant" else \
                        self.avg(self.kappa[c], i, 0) if closure == "amd" else self.avg(self.nu, i, 0) / s["closure"][3]
                    dif.append(self.diff(self.area(i) * self.flux(-kappa * self.grad(f[c], i, 0, ()), (i,)), i, 1, (i,)))
            out[c] = -sum(adv) / volume - (sum(dif) / volume if dif else 0)
        if s["flat"]:
            out["w"] = torch.zeros_like(f["w"])
        return out

    # ---- pressure
    def divergence(self):
        vel = {X: "u", Y: "v", Z: "w"}
        return sum(self.diff(self.f[vel[a]], a, 1, (a,)) / self.spacing(a, False) for a in self.axes)

    def invert(self, b):
        """∇²x = b without the bottom: Fourier in the periodic axes, the eigenvectors of the second
        difference between two walls."""
        nx, ny, nz = self.n
        lam = lambda n, d: (2 * torch.sin(math.pi * torch.arange(n, dtype=torch.float64, device=DEVICE) / n) / d) ** 2  # noqa: E731
        r = torch.fft.rfftn(b, dim=(Y, X))
        den = -(lam(nx, self.d[X])[None, None, :nx // 2 + 1] + lam(ny, self.d[Y])[None, :, None])
        if self.bounded:
            if "modes" not in self.masks:
                w, g = self.dzc[self.cells, 0, 0], 1 / self.dzf[self.h + 1:self.h + nz, 0, 0]
                T = torch.diag(torch.cat([-g, g[:0].new_zeros(1)]) + torch.cat([g[:0].new_zeros(1), -g])) + torch.diag(g, 1) + torch.diag(g, -1)
                e, Q = torch.linalg.eigh(T / (w.sqrt()[:, None] * w.sqrt()[None, :]))
                e[-1] = 0.0
                self.masks["modes"] = (e, Q / w.sqrt()[:, None], (Q * w.sqrt()[:, None]).T.contiguous())
            e, back, there = self.masks["modes"]
            apply = lambda M, a: torch.view_as_complex((M @ torch.view_as_real(a).reshape(nz, -1)).reshape(*a.shape, 2))  # noqa: E731
            den = den + e[:, None, None]
            den[-1, 0, 0] = 1.0
            r = apply(there, r) / den
            r[-1, 0, 0] = 0
            r = apply(back, r)
        else:
            if not self.s["flat"]:
                r = torch.fft.fft(r, dim=Z)
                den = den - lam(nz, float(self.dzc[0]))[:, None, None]
            den[0, 0, 0] = 1.0
            r = r / den
            r[0, 0, 0] = 0
            if not self.s["flat"]:
                r = torch.fft.ifft(r, dim=Z)
        x = torch.fft.irfftn(r, s=(ny, nx), dim=(Y, X))
        return x - x.mean()

    def conjugate(self, b):
        """V∇²x = b on the active cells, by preconditioned conjugate gradients down to rounding."""
        act = (~self.inactive).double()
        h, nz = self.h, self.n[2]
        V = self.d[X] * self.d[Y] * self.dzc

        def A(x):
            r = 0
            for a in self.axes:
                F = self.area(a) * act * self.at(act, a, -1) * (x - self.at(x, a, -1)) / self.spacing(a, True)
                r = r + self.at(F, a, 1) - F
            return r

        def M(r):
            z = torch.zeros_like(r)
            z[h:h + nz] = self.invert((r / V)[h:h + nz])
            return z * act

        fix = lambda r: (r - (r * act).sum() / act.sum()) * act  # noqa: E731
        r = fix(b * act)
        x, p, rho, goal = torch.zeros_like(r), None, 1.0, 1e-13 * float(r.norm())
        for _ in range(60):
            z = M(r)
            new = (r * z).sum()
            p = z if p is None else z + new / rho * p
            rho, q = new, A(p)
            alpha = rho / (p * q).sum()
            x, r = x + alpha * p, fix(r - alpha * q)
            if float(r.norm()) <= goal:
                break
        return x

    def project(self, dt):
        if self.immersed:
            for a, c in ((X, "u"), (Y, "v"), (Z, "w")):
                self.f[c] = self.flux(self.f[c], (a,))
        self.fill()
        d = self.divergence()
        p = torch.zeros_like(self.p)
        if self.immersed:
            p = self.conjugate(d * self.d[X] * self.d[Y] * self.dzc)
        else:
            p[self.cells] = self.invert(d[self.cells])
        self.copy_halo(p)
        inner = slice(self.h, self.h + self.n[2])
        for a, c in ((X, "u"), (Y, "v"), (Z, "w")):
            if a in self.axes:
                self.f[c][inner] -= (self.diff(p, a, 0, ()) / self.spacing(a, True))[inner]
        self.p = p / dt

    # ---- a step (the low-storage third-order Runge-Kutta scheme)
    def step(self, dt):
        nz, before = self.n[2], None
        for gamma, zeta in ((8 / 15, 0.0), (5 / 12, -17 / 60), (3 / 4, -5 / 12)):
            for c, (lo, hi) in self.s["flux"].items():
                if lo is not None:
                    self.G[c][self.h] += lo / self.dzc[self.h]
                if hi is not None:
                    self.G[c][self.h + nz - 1] -= hi / self.dzc[self.h + nz - 1]
            for c, a in self.f.items():
                k = slice(self.h + (1 if c == "w" and self.bounded else 0), self.h + nz)
                a[k] += dt * (gamma * self.G[c][k] + (zeta * before[c][k] if before else 0))
            self.project(dt * (gamma + zeta))
            before = self.G
            self.update()


def exact(case, seed):
    outs = []
    for m, n in enumerate(_sizes(case)):
        s = _setup(case["flow"], n)
        flow = _Flow(s, _inputs(s, case["precision"], seed, m))
        nz, h = n[2], flow.h
        if flow.immersed:
            flow.project(1.0)
        flow.update()
        for _ in range(case["steps"] if case["call"] != "update_state" else 0):
            flow.step(_setup(case["flow"], _sizes(case)[0])["dt"])
        if case["call"] == "update_state":
            out = {"G" + c: g[h + (1 if c == "w" and flow.bounded else 0):h + nz] for c, g in flow.G.items()}
            out["nu"] = flow.nu[h:h + nz]
            out.update({"kappa_" + c: a[h:h + nz] for c, a in flow.kappa.items()})
        else:
            out = {c: a[h:h + nz + (1 if c == "w" and flow.bounded else 0)] for c, a in flow.f.items()}
            if case["call"] == "time_step" and not flow.immersed:
                out["p"] = flow.p[h:h + nz]
        outs.append(out)
    return outs if case["call"] == "ensemble" else outs[0]
