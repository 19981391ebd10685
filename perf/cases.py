"""The work that is measured: scenes stepped through the public entry points of the PPPM solver.

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` one more of the same
ranges, `prepare(case, seed)` what a program has in hand before the call (handles with their meshes
set, inputs on the GPU), `run(state)` one pass, `work(case)` the bytes and operations the pass cannot
do without, `tolerance(case)` how far a correct implementation may be off, and `exact(case, seed)`
the same outputs in 64 bits, from plain torch.

Kinds of case:
  step           the per-sample loop body: one update_grid_and_face call, one listener read
  static         a clip on a static mesh: reset, then `run` over all steps
  moving         a clip with a moving mesh: `run_moving`, or (host) update_mesh_and_step per sample
  setup          a new mesh on a handle (every weight from scratch) and the clip's first samples
  batch          many uneven scenes stepped together
  adjoint        loss and gradient of one scene with checkpoints
  batch_adjoint  the same for several scenes together
  modal          surface accelerations of a vibrating body, a block of audio samples per call
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pppm-tdbem_amd"))
import autograd as pppm_autograd  # noqa: E402
import pppm_amd  # noqa: E402
import scenes  # noqa: E402

C = 343.0       # speed of sound
RC = 0.83       # reflection coefficient of the solver
RADIUS = 0.05   # object size of every scene (m)
KINDS = ("step", "static", "moving", "setup", "batch", "adjoint", "batch_adjoint", "modal")


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the demo's loop body on its plain scene: one sample per call, inputs from the host
        {"name": "step_32_host", "kind": "step", "res": 32, "level": 3, "extent": 2.0, "host": True},
        # the plain static scene (32^3 over two diameters of a 1280-triangle sphere), a short clip
        {"name": "static_32", "kind": "static", "res": 32, "level": 3, "extent": 2.0, "steps": 64, "listeners": 1},
        # the default grid of a finely meshed object, several listeners
        {"name": "static_64", "kind": "static", "res": 64, "level": 4, "extent": 2.0, "steps": 64, "listeners": 3},
        # an odd edge past the small-grid range, a wider margin around the object
        {"name": "static_141", "kind": "static", "res": 141, "level": 5, "extent": 3.0, "steps": 32, "listeners": 2},
        # one grid beyond every cache: the pressure stream dominates
        {"name": "static_512", "kind": "static", "res": 512, "level": 5, "extent": 8.0, "steps": 16, "listeners": 1},
        # a moving sphere beside a static cube, the mesh updated before every sample
        {"name": "moving_64", "kind": "moving", "res": 64, "level": 4, "cube": 3, "steps": 20, "host": False},
        # the same on a small odd grid, sample by sample from host buffers
        {"name": "moving_39_host", "kind": "moving", "res": 39, "level": 2, "cube": 1, "steps": 8, "host": True},
        # a new object in a fine grid: geometry, lists and every quadrature, then the first samples
        {"name": "setup_128", "kind": "setup", "res": 128, "level": 5, "extent": 2.0, "steps": 4},
        # 64 uneven scenes (24..96 cells an edge, 80..5120 triangles) stepped together
        {"name": "batch_64", "kind": "batch", "scenes": 64, "sizes": 20261205, "steps": 32},
        # loss and gradient of one scene with sqrt(T) checkpoints
        {"name": "adjoint_48", "kind": "adjoint", "res": 48, "level": 3, "extent": 2.0, "steps": 144, "listeners": 2},
        # source reconstruction over several scenes: one descent step's loss and gradients
        {"name": "batch_adjoint_64", "kind": "batch_adjoint", "scenes": 4, "res": 64, "level": 5, "extent": 2.0,
         "steps": 36, "listeners": 8},
        # surface accelerations of a modal body, a block of audio samples
        {"name": "modal_20480", "kind": "modal", "triangles": 20480, "modes": 200, "samples": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _level(rng, res, extent, top=5):
    """An icosphere level the grid resolves: about one triangle per surface cell up to sixteen."""
    across = res / extent  # cells across the object
    fits = [v for v in range(1, top + 1) if 0.1 <= 20 * 4 ** v / (math.pi * across * across) <= 16.0]
    return rng.choice(fits) if fits else 1


def draw(rng):
    """One more case. Clips that would cost more than the largest listed one are shortened."""
    kind = rng.choices(KINDS, (2, 5, 4, 2, 3, 2, 2, 2))[0]
    if kind == "modal":
        return {"kind": kind, "triangles": _log(rng, 80, 20480), "modes": _log(rng, 10, 200),
                "samples": _log(rng, 64, 1024)}
    if kind == "batch":
        case = {"kind": kind, "scenes": _log(rng, 3, 64), "sizes": rng.randrange(1 << 20), "steps": _log(rng, 8, 48)}
    elif kind == "moving":
        res = _log(rng, 28, 72)
        case = {"kind": kind, "res": res, "level": rng.choice((2, 3) if res < 48 else (3, 4)),
                "cube": rng.choice((1, 2, 3)), "steps": _log(rng, 6, 24), "host": rng.random() < 0.4}
    else:
        top = {"static": 400, "step": 160, "setup": 160, "adjoint": 72, "batch_adjoint": 64}[kind]
        res, extent = _log(rng, 24, top), round(rng.uniform(2.0, 4.0), 2)
        case = {"kind": kind, "res": res, "level": _level(rng, res, extent, 4 if kind == "adjoint" else 5),
                "extent": extent}
        if kind == "step":
            case["host"] = rng.random() < 0.5
        elif kind == "setup":
            case["steps"] = rng.randint(1, 4)
        else:
            case.update(steps=_log(rng, 12, 100), listeners=rng.randint(1, 8))
        if kind == "batch_adjoint":
            case["scenes"] = rng.randint(2, 4)
    most = max(work(c)["bytes"] for c in listed())
    while case.get("steps", 1) > 1 and work(case)["bytes"] > most:
        case["steps"] -= 1
    return case


# ------------------------------------------------------------------------------------ inputs
_SPHERES, _PAIRS = {}, {}


def _sphere(level):
    """The unit icosphere of a level (made once: the subdivision is a Python loop)."""
    if level not in _SPHERES:
        _SPHERES[level] = scenes.icosphere(level, 1.0)
    return _SPHERES[level]


class Scene:
    """Grid and mesh of one object: a sphere stretched by up to a fifth along each axis, each
    vertex's radius scaled by up to 2 %, in a cubic grid `extent` times its longest side."""

    def __init__(self, res, level, extent, seed):
        rng = np.random.default_rng(seed)
        v, f = _sphere(level)
        v = v.astype(np.float64) * RADIUS * (1 + rng.uniform(-0.02, 0.02, (v.shape[0], 1)))
        self.verts = (v * rng.uniform(0.8, 1.2, 3)).astype(np.float32)
        self.tris = f
        lo, hi = self.verts.min(0).astype(np.float64), self.verts.max(0).astype(np.float64)
        length = extent * float((hi - lo).max())
        self._grid(res, np.float32(length / res), (lo + hi) / 2 - length / 2)

    def _grid(self, res, h, low):
        self.res, self.h = res, float(h)
        self.dt = float(np.float32(self.h / (math.sqrt(3.0) * C)))
        self.min_pos = np.asarray(low, np.float32)

    def solver(self):
        s = pppm_amd.PPPMSolver(self.res, self.h, self.dt, self.min_pos, 0, RC, C)
        s.set_mesh(self.verts, self.tris)
        return s

    def listeners(self, n, seed):
        """n distinct cells a few cells off the object's surface, clear of the boundary."""
        rng, got, tries = np.random.default_rng(seed + 1), [], 0
        mid = (self.verts.min(0) + self.verts.max(0)) / 2
        while len(got) < n:
            v = self.verts[rng.integers(len(self.verts))]
            out = (v - mid) / np.linalg.norm(v - mid)
            tries += 1
            q = (v - self.min_pos) / self.h + out * rng.uniform(2.5, 6.0 + tries / 100)
            cell = tuple(int(x) for x in np.clip(q.astype(int), 3, self.res - 4))
            if cell not in got:
                got.append(cell)
        return got


class MovingScene(Scene):
    """A static cube (side 0.08 m) and a sphere (radius 0.05 m) in a cubic grid of 0.32 m; the sphere
    moves along x (0.3 cells, 200 Hz, seen around its peak velocity) and turns at 2 rad/s."""

    def __init__(self, res, level, cube, seed):
        rng = np.random.default_rng(seed)
        cv, cf = scenes.subdivided_cube(cube, side=0.08, center=(-0.07, 0.0, 0.0))
        sv, sf = _sphere(level)
        self.cube_v, self.sphere_v = cv, sv.astype(np.float64) * RADIUS
        self.tris = np.concatenate([cf, sf + cv.shape[0]]).astype(np.int32)
        self._grid(res, np.float32(0.32 / res), (-0.16, -0.16, -0.16))
        axis = rng.standard_normal(3)
        self.axis, self.start = axis / np.linalg.norm(axis), rng.uniform(-40, 40)
        self.verts = self.at(-1)

    def at(self, step):
        t = (self.start + step) * self.dt
        k = np.array([[0, -self.axis[2], self.axis[1]], [self.axis[2], 0, -self.axis[0]],
                      [-self.axis[1], self.axis[0], 0]])
        r = np.eye(3) + math.sin(2 * t) * k + (1 - math.cos(2 * t)) * (k @ k)
        off = np.array([0.07 + 0.3 * self.h * math.sin(2 * math.pi * 200.0 * t), 0.0, 0.0])
        return np.concatenate([self.cube_v, self.sphere_v @ r.T + off]).astype(np.float32)


def _accelerations(steps, nt, dt, seed):
    """(steps, nt) surface accelerations on the GPU: per triangle a tone of 0.5 to 4 kHz of its own
    phase and strength."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    freq, phase, amp = torch.rand(3, 1, nt, generator=g, device="cuda")
    t = torch.arange(steps, device="cuda", dtype=torch.float32)[:, None] * dt
    return (amp + 0.5) * torch.sin(2 * math.pi * ((500.0 + 3500.0 * freq) * t + phase))


class _Memory:
    """A solver's device memory as a tensor; the tensor keeps the handle alive."""

    def __init__(self, solver, ptr, shape):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "version": 2, "strides": None}


def _pressure(solver):
    """The current pressure level, in place."""
    return torch.as_tensor(_Memory(solver, solver.grid_ptr(0), (solver.res(),) * 3), device="cuda")


def _surface(solver):
    """The surface pressures of the last 32 steps (a ring per triangle), in place."""
    import ctypes
    n, d = ctypes.c_void_p(), ctypes.c_void_p()
    if solver.lib.pppm_history_ptrs(solver.h, ctypes.byref(n), ctypes.byref(d)) != 0:
        raise pppm_amd.PPPMError("history_ptrs failed")
    return torch.as_tensor(_Memory(solver, d.value, (solver.nt, 32)), device="cuda")


def _field(solver):
    return {"pressure": _pressure(solver), "surface": _surface(solver)}


def _batch_scenes(case, seed):
    sizes = scenes.c3_batch_sizes(case["scenes"], case["sizes"])
    return [Scene(r, v, 2.0, seed * 1009 + i) for i, (r, v) in enumerate(sizes)]


def _modal_inputs(case, seed):
    rng = np.random.default_rng(seed)
    nt, modes = case["triangles"], case["modes"]
    nv = nt // 2 + 2
    normals = rng.standard_normal((nt, 3))
    freq = np.sort(rng.uniform(100.0, 15000.0, modes))
    return {"eig": (rng.standard_normal((3 * nv, modes), dtype=np.float32) * np.float32(0.1)),
            "eigvals": ((2 * np.pi * freq) ** 2).astype(np.float32),
            "tris": rng.integers(0, nv, (nt, 3)).astype(np.int32),
            "normals": (normals / np.linalg.norm(normals, axis=1, keepdims=True)).astype(np.float32),
            "forces": rng.standard_normal((case["samples"], modes), dtype=np.float32) * np.float32(1e3)}


MATERIAL = (30.0, 1e-6, 44100.0)  # Rayleigh damping of the modal body, its sample rate
WARM = 40                         # samples a `step` case's handle has behind it


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind == "modal":
        x = _modal_inputs(case, seed)
        st["source"] = pppm_amd.ModalSource(x["eig"], x["eigvals"], x["tris"], x["normals"], *MATERIAL)
        st["forces"] = torch.from_numpy(x["forces"]).cuda()
        st["accs"] = torch.empty(case["samples"], case["triangles"], device="cuda")
        return st
    if kind in ("batch", "batch_adjoint"):
        sc = (_batch_scenes(case, seed) if kind == "batch" else
              [Scene(case["res"], case["level"], case["extent"], seed * 1009 + i) for i in range(case["scenes"])])
        n = case.get("listeners", 1)
        st["solvers"] = [s.solver() for s in sc]
        st["batch"] = pppm_amd.PPPMBatch(st["solvers"])
        st["listeners"] = [s.listeners(n, seed) for s in sc]
        st["inputs"] = [_accelerations(case["steps"], len(s.tris), s.dt, seed * 1009 + i) for i, s in enumerate(sc)]
        if kind == "batch":
            st["out"] = torch.zeros(case["steps"], len(sc), n, device="cuda")
        else:
            st["targets"] = [_target(case, seed * 1009 + i) for i in range(len(sc))]
        return st
    if kind == "moving":
        sc = MovingScene(case["res"], case["level"], case["cube"], seed)
        st["solver"] = sc.solver()
        verts = np.stack([sc.at(i) for i in range(case["steps"])])
        acc = _accelerations(case["steps"], len(sc.tris), sc.dt, seed)
        st["listeners"] = sc.listeners(1, seed)
        if case["host"]:
            st["verts"], st["inputs"] = verts, acc.cpu().numpy()
        else:
            st["verts"], st["inputs"] = torch.from_numpy(verts).cuda(), acc
            st["out"] = torch.zeros(case["steps"], 1, device="cuda")
        return st
    sc = Scene(case["res"], case["level"], case["extent"], seed)
    st["solver"] = sc.solver()
    st["listeners"] = sc.listeners(case.get("listeners", 1), seed)
    if kind == "step":
        acc = _accelerations(WARM + 64, len(sc.tris), sc.dt, seed)
        st["solver"].run(acc[:WARM].contiguous(), WARM, [], None)
        torch.cuda.synchronize()
        st["rows"] = list(acc[WARM:].cpu().numpy() if case["host"] else acc[WARM:])
        st["next"] = 0
        return st
    st["inputs"] = _accelerations(case["steps"], len(sc.tris), sc.dt, seed)
    if kind == "adjoint":
        st["target"] = _target(case, seed)
    else:
        st["out"] = torch.zeros(case["steps"], len(st["listeners"]), device="cuda")
    if kind == "setup":
        st["verts"], st["tris"] = torch.from_numpy(sc.verts).cuda(), torch.from_numpy(sc.tris).cuda()
    return st


def _target(case, seed):
    """Listener samples to fit: a tone at the strength of the listeners' own signal."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 7)
    phase = torch.rand(1, case["listeners"], generator=g, device="cuda")
    t = torch.arange(case["steps"], device="cuda", dtype=torch.float32)[:, None] / case["steps"]
    return 1e-3 * t * torch.sin(2 * math.pi * (3 * t + phase))


# ------------------------------------------------------------------------------------ one pass
def run(st):
    kind = st["kind"]
    if kind == "step":
        s = st["solver"]
        s.update_grid_and_face(st["rows"][st["next"] % len(st["rows"])])
        st["next"] += 1
        return dict(_field(s), sample=s.read_cells(st["listeners"]))
    if kind == "static":
        s = st["solver"]
        s.reset()
        s.run(st["inputs"], st["case"]["steps"], st["listeners"], st["out"])
        return dict(_field(s), samples=st["out"])
    if kind == "moving":
        s, n = st["solver"], st["case"]["steps"]
        s.reset()
        if st["case"]["host"]:
            samples = np.zeros((n, 1), np.float32)
            for i in range(n):
                s.update_mesh_and_step(st["verts"][i], st["inputs"][i])
                samples[i] = s.read_cells(st["listeners"])
        else:
            samples = st["out"]
            s.run_moving(st["verts"], st["inputs"], n, st["listeners"], samples)
        return dict(_field(s), samples=samples)
    if kind == "setup":
        s = st["solver"]
        s.set_mesh(st["verts"], st["tris"])
        s.reset()
        s.run(st["inputs"], st["case"]["steps"], st["listeners"], st["out"])
        return dict(_field(s), samples=st["out"])
    if kind == "batch":
        for s in st["solvers"]:
            s.reset()
        st["batch"].run(st["inputs"], st["case"]["steps"], st["listeners"], st["out"])
        some = st["solvers"][:: max(1, len(st["solvers"]) // 24)][:24]  # fields of up to 24 scenes
        return {"samples": st["out"], "fields": [_field(s) for s in some]}
    if kind == "adjoint":
        g = st["inputs"].detach().requires_grad_()
        loss = pppm_autograd.listener_loss(g, st["target"], st["solver"], st["listeners"])
        loss.backward()
        return {"loss": loss.detach(), "gradient": g.grad}
    if kind == "batch_adjoint":
        gs = [g.detach().requires_grad_() for g in st["inputs"]]
        loss = pppm_autograd.batch_listener_loss(st["batch"], st["solvers"], gs, st["targets"], st["listeners"])
        loss.sum().backward()
        return {"loss": loss.detach(), "gradients": [g.grad for g in gs]}
    st["source"].run(st["forces"], st["accs"])
    return {"accelerations": st["accs"]}


# ------------------------------------------------------------------------------------ work
def _pair_counts(key, make):
    """(triangles, corrected cells, cell pairs, face pairs) of a mesh in its grid, from the
    triangles' cells: the cells within one of a triangle's, and the triangles in the 4x4x4 cells
    around each triangle's base cell."""
    if key not in _PAIRS:
        v, f, low, h = make()
        ctr = v[f].mean(1)
        cell = np.floor((ctr - low) / h).astype(int)
        base = np.floor((ctr - low) / h - 0.5).astype(int)
        first = cell.min(0)
        cell, base = cell - first, base - first
        span = int(cell.max()) + 1
        count = np.zeros((span + 8,) * 3, np.int64)
        np.add.at(count, tuple((cell + 4).T), 1)
        total = np.zeros((span + 9,) * 3, np.int64)
        total[1:, 1:, 1:] = count.cumsum(0).cumsum(1).cumsum(2)

        def box(lo, hi):  # triangles in the cells lo..hi - 1 of each row
            lo, hi = lo + 4, hi + 4
            s = 0
            for m in range(8):
                q = [hi[:, d] if m >> d & 1 else lo[:, d] for d in range(3)]
                s = s + (1 if bin(m).count("1") % 2 else -1) * total[q[0], q[1], q[2]]
            return s
        p4 = int(box(base - 1, base + 3).sum())
        near = np.unique(np.concatenate([cell + np.array(o) for o in np.ndindex(3, 3, 3)]) - 1, axis=0)
        _PAIRS[key] = (len(f), len(near), 27 * len(f), p4)
    return _PAIRS[key]


def _static_counts(res, level, extent):
    def make():
        v, f = _sphere(level)
        length = extent * 2 * RADIUS
        return v.astype(np.float64) * RADIUS, f, -length / 2, length / res
    return _pair_counts(("static", res, level, extent), make)


def _step_work(res, counts, host=False):
    """One time step: three pressure levels, a weight record, its scales and its index per pair, the
    corrected cells, the triangles' histories and results; 16 taps of two fields per pair."""
    nt, c3, p3, p4 = counts
    b = 12.0 * res ** 3 + 152.0 * p3 + 16.0 * c3 + 76.0 * p4 + 204.0 * nt
    return b, 12.0 * res ** 3 + 96.0 * (2 * p3 + p4)


def work(case):
    kind = case["kind"]
    if kind == "modal":
        nt, m, s = case["triangles"], case["modes"], case["samples"]
        return {"bytes": 4.0 * (nt * m + s * m + s * nt), "flops": 2.0 * nt * m * s}
    if kind == "batch":
        per = [_step_work(r, _static_counts(r, v, 2.0)) for r, v in scenes.c3_batch_sizes(case["scenes"], case["sizes"])]
        b, f = (case["steps"] * sum(p[i] for p in per) for i in (0, 1))
    elif kind == "moving":
        def make():
            m = MovingScene(case["res"], case["level"], case["cube"], 0)
            return m.verts.astype(np.float64), m.tris, -0.16, 0.32 / case["res"]
        counts = _pair_counts(("moving", case["res"], case["level"], case["cube"]), make)
        b, f = _step_work(case["res"], counts)
        # each update: vertices and triangles in, geometry, cells, lists and interpolation weights out
        nt, c3, p3, p4 = counts
        b, f = (b + 160.0 * nt + 4.0 * (p3 + p4) + 8.0 * c3) * case["steps"], f * case["steps"]
    else:
        counts = _static_counts(case["res"], case["level"], case["extent"])
        b, f = _step_work(case["res"], counts)
        steps = case.get("steps", 1) * case.get("scenes", 1)
        if kind in ("adjoint", "batch_adjoint"):
            # forward, recomputed forward, transposed step (16 B a cell), gradient rows
            b, f = 3 * b + 4.0 * case["res"] ** 3 + 4.0 * counts[0], 3 * f
        b, f = b * steps, f * steps
        if kind == "setup":
            # weights out; 81 targets of 9 wave numbers per triangle, one point pair per face pair
            nt, c3, p3, p4 = counts
            b, f = b + 148.0 * p3 + 80.0 * p4, f + 1.6e5 * nt + 6e3 * p4
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------------------------ tolerances
def tolerance(case):
    """About four times the largest distance of the outputs from exact() over the declared ranges:
    1.2e-5 for pressures, surface values and gradients of 32-bit sums, 3e-5 to 5e-5 for the second
    differences of 32-bit oscillator positions."""
    return {"rel": 2e-4 if case["kind"] == "modal" else 5e-5}


# ------------------------------------------------------------------------------------ 64 bits
PI = 3.14159265359  # the constant of the solver's definition
TAPS = 16


def _cplx(re, im):
    return torch.complex(re, im)


class Exact:
    """The PPPM step of a static scene in float64 (weights: float64 quadrature, stored as 16-bit
    codes with a 32-bit scale per series, as the solver defines them)."""

    def __init__(self, sc):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.n, self.h, self.dt = sc.res, sc.h, sc.dt
        f32 = np.float32
        v, f = sc.verts, sc.tris
        low = sc.min_pos
        # cells and base cells are decided on 32-bit centres
        ctr = ((v[f[:, 0]] + v[f[:, 1]] + v[f[:, 2]]) / f32(3.0)).astype(f32)
        cell = ((ctr - low) / f32(sc.h)).astype(np.int32)
        mid = (cell.astype(f32) + f32(0.5)) * f32(sc.h) + low
        base = cell - (ctr - mid < 0)
        self.ctr32 = ctr
        t64 = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=self.dev)  # noqa: E731
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64, device=self.dev)  # noqa: E731
        self.low, self.cell, self.base, self.idx = t64(low), t(cell), t(base), t(f)
        self.V = t64(v)[self.idx]  # (T, 3, 3)
        cr = torch.cross(self.V[:, 1] - self.V[:, 0], self.V[:, 2] - self.V[:, 0], dim=1)
        self.jac = cr.norm(dim=1)
        self.nrm = cr / self.jac[:, None]
        self.pt = self.V.sum(1) / 3
        # wave numbers and the inverse transform with its scaling
        cdt = self.dt * C
        lam = max(cdt ** (3.0 / TAPS), float(f32(1e-8)) ** (1.0 / (2 * TAPS)))
        s = lam * np.exp(-2j * PI / TAPS * np.arange(9))
        wave = 1j * (0.5 * (s * s - 4 * s + 3) / cdt)
        self.wave = torch.as_tensor(wave, dtype=torch.complex128, device=self.dev)
        m = np.exp(2j * PI / TAPS * np.outer(np.arange(9), np.arange(TAPS))) / TAPS * lam ** -np.arange(TAPS)
        m[1:8] *= 2  # wave numbers 9..15 are the conjugates of 7..1
        self.idft = torch.as_tensor(m, dtype=torch.complex128, device=self.dev)
        self._interp()
        self._grid_weights()
        self._face_weights()
        self._boundary()

    def _centre(self, cell):
        return (cell.double() + 0.5) * self.h + self.low

    def _layers(self, src, trg, nrm):
        """Both layer kernels at the nine wave numbers: (..., 9) each; 0 where the points coincide."""
        d = src - trg
        r2 = (d * d).sum(-1)
        r = r2.sqrt().clamp_min(1e-300)
        ikr = 1j * r[..., None] * self.wave
        e = ikr.exp()
        single = e / (4 * PI * r)[..., None]
        dn = (d * nrm).sum(-1)
        double = -e * (1 - ikr) * (dn / (4 * PI * r2.clamp_min(1e-300) * r))[..., None]
        on = (r2 > 0)[..., None]
        return torch.where(on, single, 0 * single), torch.where(on, double, 0 * double)

    def _series(self, x):
        return (x @ self.idft).real

    @staticmethod
    def _stored(w):
        """16-bit codes over the series' largest value, as float64."""
        top = w.float().abs().amax(-1, keepdim=True)
        top = torch.where(top == 0, torch.ones_like(top), top)
        return (w.float() / top).half().double() * top.double()

    def _interp(self):
        d = (self.pt - self._centre(self.base)) / self.h
        w = []
        for k in range(8):
            q = [d[:, a] if (k >> (2 - a)) & 1 else 1 - d[:, a] for a in range(3)]
            w.append(q[0] * q[1] * q[2])
        self.interp = (0.5 * self.jac)[:, None] * torch.stack(w, 1)
        off = torch.tensor([[k >> 2 & 1, k >> 1 & 1, k & 1] for k in range(8)], device=self.dev)
        self.corner_cells = self.base[:, None] + off
        self.corners = self._lin(self.corner_cells)

    def _lin(self, c):
        return (c[..., 0] * self.n + c[..., 1]) * self.n + c[..., 2]

    def _grid_weights(self):
        """Per (triangle, neighbour cell): the correction of the stencil and of the cell itself."""
        T, dev = len(self.cell), self.dev
        scale = float(np.float32(C) ** 2 * np.float32(self.dt) ** 2 / np.float32(self.h) ** 2)
        around = torch.tensor([[x, y, z] for x in range(-2, 3) for y in range(-2, 3) for z in range(-2, 3)], device=dev)
        at = lambda o: ((o[..., 0] + 2) * 5 + o[..., 1] + 2) * 5 + o[..., 2] + 2  # noqa: E731
        own = int(at(torch.zeros(3, dtype=torch.long)))
        offs = torch.tensor([[o % 3 - 1, o // 3 % 3 - 1, o // 9 - 1] for o in range(27)], device=dev)
        step = torch.tensor([[0, 0, 0], [-1, 0, 0], [1, 0, 0], [0, -1, 0], [0, 1, 0], [0, 0, -1], [0, 0, 1]], device=dev)
        S = torch.zeros(125, 27, dtype=torch.float64, device=dev)  # stencil of each offset over the 125 cells
        for o in range(27):
            for k in range(7):
                S[at(offs[o] + step[k]), o] += (2 - 6 * scale) if k == 0 else scale
        S[own] = 0  # the triangle's own cell is left out
        one = torch.zeros(125, 27, dtype=torch.float64, device=dev)
        for o in range(27):
            one[at(offs[o]), o] = 1
        one[own] = 0
        self.wf, self.wb = [], []
        for a in range(0, T, 2048):
            b = min(T, a + 2048)
            trg = self._centre(self.cell[a:b, None] + around)
            layers = self._layers(self.pt[a:b, None].expand_as(trg), trg, self.nrm[a:b, None])
            f = (0.5 * self.jac[a:b])[:, None, None]
            out = []
            for g in layers:
                g = (f * g).movedim(1, 2)  # (t, 9, 125)
                sten, near = ((g @ m.to(g.dtype)).movedim(1, 2) for m in (S, one))
                sten, near = self._series(sten), self._series(near)  # (t, 27, 16)
                w = torch.zeros_like(sten)
                w[..., 1:] = sten[..., :-1]
                w[..., 2:] -= near[..., :-2]
                out.append((self._stored(w), self._stored(near)))
            self.wf.append(torch.stack([-out[0][0], out[1][0]]))
            self.wb.append(torch.stack([-out[0][1], out[1][1]]))
        self.wf, self.wb = torch.cat(self.wf, 1), torch.cat(self.wb, 1)  # (2, T, 27, 16)
        self.c3_cell = self._lin(self.cell[:, None] + offs)  # (T, 27)
        self.c3 = torch.unique(self.c3_cell)

    def _pairs(self):
        """(c, j): j's cell lies in the 4x4x4 block around c's base cell."""
        got = []
        for a in range(0, len(self.cell), 1024):
            d = self.cell[None] - self.base[a:a + 1024, None]
            c, j = ((d >= -1) & (d <= 2)).all(-1).nonzero(as_tuple=True)
            got.append(torch.stack([c + a, j]))
        return torch.cat(got, 1)

    def _singular(self, c, j, shared):
        """Sauter-Schwab rules of order 3 for pairs that share vertices; j is the trial triangle."""
        x, w = np.array([0.774596669241483, 0.0, -0.774596669241483]), np.array([0.555555555555554, 0.888888888888889, 0.555555555555554])
        p = 0.5 * (x + 1)
        xi, e1, e2, e3 = (torch.as_tensor(q.reshape(-1), device=self.dev) for q in np.meshgrid(p, p, p, p, indexing="ij"))
        w = torch.as_tensor(np.einsum("a,b,c,d->abcd", w, w, w, w).reshape(-1), device=self.dev)
        e12, e123 = e1 * e2, e1 * e2 * e3
        one = torch.ones_like(xi)
        if shared == 3:
            jw = xi ** 3 * e1 ** 2 * e2
            q = [(xi, xi * (1 - e1 + e12)), (xi * (1 - e123), xi * (1 - e1)), (xi, xi * (e1 - e12 + e123)),
                 (xi * (1 - e12), xi * (e1 - e12)), (xi * (1 - e123), xi * (e1 - e123)), (xi, xi * (e1 - e12))]
            terms = [(q[0], q[1], one), (q[1], q[0], one), (q[2], q[3], one), (q[3], q[2], one), (q[4], q[5], one),
                     (q[5], q[4], one)]
        elif shared == 2:
            jw = xi ** 3 * e1 ** 2
            terms = [((xi, xi * e1 * e3), (xi * (1 - e12), xi * e1 * (1 - e2)), one),
                     ((xi, xi * e1), (xi * (1 - e123), xi * e12 * (1 - e3)), e2),
                     ((xi * (1 - e12), xi * e1 * (1 - e2)), (xi, xi * e123), e2),
                     ((xi * (1 - e123), xi * e12 * (1 - e3)), (xi, xi * e1), e2),
                     ((xi * (1 - e123), xi * e1 * (1 - e2 * e3)), (xi, xi * e12), e2)]
        else:
            jw = xi ** 3 * e2
            terms = [((xi, xi * e1), (xi * e2, xi * e2 * e3), one), ((xi * e2, xi * e2 * e3), (xi, xi * e1), one)]

        def place(uv, v):  # (pairs, 81, 3)
            u, t = uv[0][:, None], uv[1][:, None]
            return (1 - u) * v[:, None, 0] + (u - t) * v[:, None, 1] + t * v[:, None, 2]
        s = d = 0
        for a, b, f in terms:
            gs, gd = self._layers(place(a, self.V[j]), place(b, self.V[c]), self.nrm[j][:, None])
            f = (f * jw * w)[None, :, None]
            s, d = s + (f * gs).sum(1), d + (f * gd).sum(1)
        f = (self.jac[j] * self.jac[c] / 16)[:, None]
        return f * s, f * d

    def _face_weights(self):
        c, j = self._pairs()
        ctr32 = torch.as_tensor(self.ctr32, device=self.dev)
        shared = (self.idx[c][:, :, None] == self.idx[j][:, None, :]).sum((1, 2))
        close = (ctr32[c] - ctr32[j]).norm(dim=1) < float(np.float32(self.h * 0.1))
        wf = []
        for a in range(0, len(c), 1 << 16):
            q = slice(a, a + (1 << 16))
            cc, jj, sh, cl = c[q], j[q], shared[q], close[q]
            s, d = self._layers(self.pt[jj], self.pt[cc], self.nrm[jj])
            f = (0.25 * self.jac[jj] * self.jac[cc])[:, None] * (~cl)[:, None]
            s, d = f * s, f * d
            for k in (1, 2, 3):
                at = (sh == k).nonzero()[:, 0]
                for b in at.split(2048):
                    if len(b):
                        s[b], d[b] = self._singular(cc[b], jj[b], k)
            # the far field the grid already carries: the corners of c's base cell not near j
            ctr = self._centre(self.corner_cells[cc])  # (p, 8, 3)
            mid32 = (self.corner_cells[cc].float() + 0.5) * self.h + self.low.float()  # decided on 32-bit centres
            far = ((mid32 - ctr32[jj][:, None]).abs().double() > self.h * 1.5).any(-1)
            gs, gd = self._layers(self.pt[jj][:, None].expand_as(ctr), ctr, self.nrm[jj][:, None])
            wt = (torch.where(far, -self.interp[cc], torch.zeros_like(far, dtype=torch.float64)) *
                  (0.5 * self.jac[jj])[:, None])[..., None]
            s, d = s + (wt * gs).sum(1), d + (wt * gd).sum(1)
            wf.append(torch.stack([-self._stored(self._series(s)), self._stored(self._series(d))]))
        self.pc, self.pj, self.pw = c, j, torch.cat(wf, 1)  # (2, P, 16)
        lump = torch.zeros(len(self.cell), dtype=torch.float64, device=self.dev).index_add(0, c, self.pw[1, :, 0])
        self.den = 0.25 * self.jac - lump

    def _boundary(self):
        """The first-order absorbing condition: one 4x4 system per cell of the outer shell."""
        n, h, dt = self.n, self.h, self.dt
        r = torch.arange(1, n - 1, device=self.dev)
        sel = torch.zeros(n - 2, n - 2, n - 2, dtype=torch.bool, device=self.dev)
        for d in range(3):
            sel.select(d, 0).fill_(True)
            sel.select(d, n - 3).fill_(True)
        co = torch.stack([r[i] for i in sel.nonzero(as_tuple=True)], 1)
        judge = (co == n - 2).long() - (co == 1).long()
        k0, k1, k2, k3 = C * C * dt * dt / (h * h), 1 / (dt * dt), C / (2 * h * dt), -C * C / (2 * h * h)
        at = (judge != 0).double()
        A = torch.zeros(len(co), 4, 4, dtype=torch.float64, device=self.dev)
        A[:, 3, 3] = 1
        for x in range(3):
            y, z = (x + 1) % 3, (x + 2) % 3
            A[:, 3, x] = -k0 * at[:, x]
            A[:, x, 3], A[:, x, x] = k1, k2
            A[:, x, y], A[:, x, z] = k3 * at[:, y], k3 * at[:, z]
        kinds, which = torch.unique((at.long() * torch.tensor([1, 2, 4], device=self.dev)).sum(1), return_inverse=True)
        first = torch.stack([(which == q).nonzero()[0, 0] for q in range(len(kinds))])
        self.ainv = torch.linalg.inv(A[first])[which]
        self.shell, self.judge, self.k = self._lin(co), judge, (k0, k1, k2, k3)
        strd = torch.tensor([n * n, n, 1], device=self.dev)
        self.strd = strd
        self.ghost_row, self.ghost_dir = judge.nonzero(as_tuple=True)
        self.ghost = self.shell[self.ghost_row] + (judge * strd)[self.ghost_row, self.ghost_dir]

    def _fdtd(self, old, prev, cur):
        """(cur with its ghost layer, next level): the next level overwrites the oldest one."""
        n, (k0, k1, k2, k3) = self.n, self.k
        m, i = slice(2, n - 2), [slice(1, n - 3), slice(3, n - 1)]
        lap = -6 * cur[m, m, m]
        for q in i:
            lap = lap + cur[q, m, m] + cur[m, q, m] + cur[m, m, q]
        new = old.clone()
        new[m, m, m] = 2 * cur[m, m, m] - prev[m, m, m] + C * C * self.dt * self.dt / (self.h * self.h) * lap
        g, gm, me = cur.reshape(-1), prev.reshape(-1), self.shell
        gc, gmc, j = g[me], gm[me], self.judge
        up = [g[me + s] * (j[:, d] <= 0) for d, s in enumerate(self.strd)]
        dn = [g[me - s] * (j[:, d] >= 0) for d, s in enumerate(self.strd)]
        rows = []
        for x in range(3):
            y, z, s = (x + 1) % 3, (x + 2) % 3, self.strd[x]
            jx = j[:, x]
            slope = (g[me + s] * -(jx < 0).double() - g[me - s] * (jx > 0).double() + gm[me + s] * -jx + gm[me - s] * jx)
            rows.append(-k1 * (gmc - 2 * gc) - k2 * slope - k3 * (up[y] + dn[y] + up[z] + dn[z] - 4 * gc))
        rows.append(-gmc + 2 * gc - k0 * 6 * gc + k0 * sum(a + b for a, b in zip(up, dn)))
        r = (self.ainv @ torch.stack(rows, 1)[..., None])[..., 0]
        flat, withghost = new.reshape(-1), g.clone()
        flat[me] = r[:, 3]
        withghost[self.ghost] = r[self.ghost_row, self.ghost_dir]
        return withghost.reshape(cur.shape), flat.reshape(cur.shape)

    def clip(self, inputs, listeners):
        """Steps from the zero state: listener samples (steps, L), the last pressure level and the
        surface pressures as the solver lays its 32-slot rings out."""
        n, T = self.n, len(self.cell)
        zero = torch.zeros(n, n, n, dtype=torch.float64, device=self.dev)
        old, prev, cur = zero, zero, zero
        N = torch.zeros(T, TAPS, dtype=torch.float64, device=self.dev)
        D, samples, surface = N, [], []
        where = torch.as_tensor([(x * n + y) * n + z for x, y, z in listeners], device=self.dev, dtype=torch.int64)
        cells, size = self.c3_cell.reshape(-1), n ** 3

        def spread(w, N, D):
            return torch.zeros(size, dtype=torch.float64, device=self.dev).index_add(
                0, cells, (w[0] * N[:, None] + w[1] * D[:, None]).sum(-1).reshape(-1))
        for row in inputs.to(self.dev).double():
            cur, new = self._fdtd(old, prev, cur)
            N = torch.cat([row[:, None], N[:, :-1]], 1)
            D = torch.cat([torch.zeros_like(D[:, :1]), D[:, :-1]], 1)
            far = new.reshape(-1) - spread(self.wf, N, D)
            face = (self.interp * far[self.corners]).sum(1)
            near = torch.zeros(T, dtype=torch.float64, device=self.dev)
            for q in range(0, len(self.pc), 1 << 20):
                q = slice(q, q + (1 << 20))
                near = near.index_add(0, self.pc[q], (self.pw[0, q] * N[self.pj[q]] + self.pw[1, q] * D[self.pj[q]]).sum(-1))
            d = (face * RC + near) / self.den
            D = torch.cat([d[:, None], D[:, 1:]], 1)
            new = far + 0.98 * spread(self.wb, N, D)
            old, prev, cur = prev, cur, new.reshape(n, n, n)
            samples.append(new[where])
            surface.append(d)
        ring = torch.zeros(32, T, dtype=torch.float64, device=self.dev)
        for k, d in list(enumerate(surface))[-32:]:
            ring[k % 32] = d.detach()
        return torch.stack(samples), cur, ring.T


def exact(case, seed):
    """In 64 bits; None for the moving scenes, whose weights are those of the positions at which each
    was last recomputed, and for scenes that take over 20 seconds this way."""
    kind = case["kind"]
    if kind == "modal":
        return _exact_modal(case, seed)
    if kind in ("moving", "batch_adjoint"):
        return None
    if kind == "batch":
        if case["scenes"] * case["steps"] > 200:
            return None
        out = []
        sc = _batch_scenes(case, seed)
        for i, s in enumerate(sc):
            x = Exact(s)
            out.append(x.clip(_accelerations(case["steps"], len(s.tris), s.dt, seed * 1009 + i), s.listeners(1, seed)))
        step = max(1, len(sc) // 24)
        return {"samples": torch.stack([o[0] for o in out], 1),
                "fields": [{"pressure": o[1], "surface": o[2]} for o in out[::step][:24]]}
    sc = Scene(case["res"], case["level"], case["extent"], seed)
    steps = case.get("steps", 1)
    _, _, _, p4 = _static_counts(case["res"], case["level"], case["extent"])
    if kind == "adjoint":
        if steps * (case["res"] ** 3 + 4 * p4) > 1.5e8:
            return None
        g = _accelerations(steps, len(sc.tris), sc.dt, seed).double().requires_grad_()
        samples, _, _ = Exact(sc).clip(g, sc.listeners(case["listeners"], seed))
        loss = ((samples - _target(case, seed).double()) ** 2).sum()
        loss.backward()
        return {"loss": loss.detach(), "gradient": g.grad}
    if p4 > 8e6:
        return None
    x, lis = Exact(sc), sc.listeners(case.get("listeners", 1), seed)
    with torch.no_grad():
        if kind == "step":
            samples, p, d = x.clip(_accelerations(WARM + 64, len(sc.tris), sc.dt, seed)[:WARM + 1], lis)
            return {"pressure": p, "surface": d, "sample": samples[-1]}
        samples, p, d = x.clip(_accelerations(steps, len(sc.tris), sc.dt, seed), lis)
    return {"pressure": p, "surface": d, "samples": samples}


def _exact_modal(case, seed):
    x = _modal_inputs(case, seed)
    alpha, beta, rate = MATERIAL
    dt = float(np.float32(1.0 / rate))
    lam = x["eigvals"].astype(np.float64)
    om = np.sqrt(lam)
    ksi = (alpha + beta * lam) / (2 * om)
    omp = om * np.sqrt(1 - ksi * ksi)
    eps, th, gam = np.exp(-ksi * om * dt), omp * dt, np.arcsin(ksi)
    c1, c2 = 2 * eps * np.cos(th), -eps ** 2
    c3 = 2 * (eps * np.cos(th + gam) - eps ** 2 * np.cos(2 * th + gam)) / (3 * om * omp)
    q1, q2 = np.zeros_like(om), np.zeros_like(om)
    acc = np.zeros((case["samples"], case["modes"]))
    for s, f in enumerate(x["forces"].astype(np.float64)):
        q0 = c1 * q1 + c2 * q2 + c3 * f
        acc[s] = (q0 + q2 - 2 * q1) / (dt * dt)
        q1, q2 = q0, q1
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    to = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    u = to(x["eig"]).reshape(-1, 3, case["modes"])
    tris = torch.as_tensor(x["tris"].astype(np.int64), device=dev)
    surf = torch.zeros(case["triangles"], case["modes"], dtype=torch.float64, device=dev)
    for k in range(3):
        surf += (u[tris[:, k]] * to(x["normals"])[:, :, None]).sum(1) / 3
    return {"accelerations": to(acc) @ surf.T}
