"""The work users have this package do, as cases that can be timed and checked.

A case is a plain dict. Three kinds of call are covered, each through the
package's public interface:

  "grid"      a Grid with its boundaries, objects, source and detectors,
              advanced by ``grid.run(steps)`` (``call="run"``) or by
              ``grid.step()`` in a loop (``call="step"``)
  "batch"     many unequal grids advanced together by ``GridBatch.run``
  "gradient"  objective and gradient with respect to a design region's
              permittivity, ``IntensityGradient.gradient``

``prepare`` builds what a program has in hand before the call (grids start
from seeded smooth fields, as a run that is continued does, so that every cell
carries a signal), ``run`` makes the call and returns the updated fields,
detector traces or gradient. ``exact`` steps the same inputs in float64 with
plain torch array operations (Yee updates, CPML, the object kinds and sources
written out from their equations).
"""

import math

import torch
import torch.nn.functional as F

import fdtd_amd as fdtd
from fdtd_amd.adjoint import IntensityGradient
from fdtd_amd.batch import GridBatch

C0 = 299792458.0
SPACING = 50e-9
DEV = "cuda"
ITEM = {"float64": 8, "float32": 4, "float32c": 5}


# ------------------------------------------------------------------- cases
def grid_case(shape, dtype, steps, **options):
    """A "grid" case; ``options`` override the defaults listed here."""
    case = dict(kind="grid", nx=shape[0], ny=shape[1], nz=shape[2], dtype=dtype, steps=steps, pml=10,
                periodic=False,      # periodic z in place of the two z faces
                material="uniform",  # uniform | noise (a value per cell) | spheres (few distinct values)
                objects="none",      # none | plain | absorbing (slab and anisotropic block) | complex
                source="point",      # point | line | plane
                detector="none",     # none | line | block
                call="run")
    case.update(options)
    return case


def listed():
    two_d = dict(periodic=True, objects="plain", source="line", detector="line")
    return [
        # the README's first simulation: a 2D grid with a line source, an
        # object and a line detector, run for a few hundred steps
        dict(grid_case((161, 97, 1), "float64", 100, **two_d), name="first_2d_run"),
        # the same grid advanced a step at a time from Python, as a program
        # that looks at the fields between steps does
        dict(grid_case((161, 97, 1), "float64", 2, call="step", **two_d), name="first_2d_step"),
        # a small 3D device with every object kind and a detector
        dict(grid_case((60, 52, 44), "float64", 50, pml=8, material="noise", objects="absorbing", detector="line"),
             name="small_3d_f64"),
        # an ordinary 3D simulation in single precision that fits the caches
        dict(grid_case((128, 128, 128), "float32", 40, material="noise"), name="cube128_f32"),
        # uneven edges, plane-wave excitation, a monitor over a whole plane
        dict(grid_case((201, 150, 97), "float32", 20, objects="plain", source="plane", detector="block"),
             name="ragged_planewave_f32"),
        # lossy materials make the fields complex
        dict(grid_case((96, 81, 64), "float64", 20, objects="complex"), name="lossy_complex128"),
        # the benchmark's grid in its three storages
        dict(grid_case((256, 256, 256), "float64", 10, pml=16, material="spheres"), name="cube256_f64"),
        dict(grid_case((256, 256, 256), "float32", 10, pml=16, material="spheres"), name="cube256_f32"),
        dict(grid_case((256, 256, 256), "float32c", 10, pml=16, material="spheres"), name="cube256_f32c"),
        # the largest single simulation: absorbing slab and anisotropic block
        dict(grid_case((512, 512, 384), "float32", 4, pml=20, objects="absorbing"), name="large_f32"),
        # a parameter sweep: unequal grids stepped together
        dict(kind="batch", count=24, low=64, high=160, dtype="float32", steps=100, pml=10, name="sweep_f32"),
        # inverse design: objective and gradient of one candidate
        dict(kind="gradient", nx=128, ny=128, nz=64, dtype="float32", steps=200, pml=12, checkpoint="sqrt",
             name="gradient_f32"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _steps(cells, budget, most):
    return max(2, min(most, int(budget / cells)))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["2d", "small", "medium", "medium", "large", "complex", "batch", "gradient"])
    if kind == "2d":
        shape = (_log_int(rng, 80, 700), _log_int(rng, 60, 500), 1)
        return grid_case(shape, rng.choice(["float64", "float32"]), rng.randint(20, 150),
                         pml=rng.randint(6, 12), periodic=True, objects=rng.choice(["none", "plain"]),
                         source=rng.choice(["point", "line"]), detector=rng.choice(["none", "line"]))
    if kind == "batch":
        low, count, dtype = rng.randint(32, 90), rng.randint(3, 24), rng.choice(["float32", "float64"])
        high = rng.randint(low + 8, 150)
        return dict(kind="batch", count=count, low=low, high=high, dtype=dtype, pml=rng.randint(6, 12),
                    steps=_steps(ITEM[dtype] * count * high ** 3, 1.3e10, rng.randint(20, 120)))
    if kind == "gradient":
        return dict(kind="gradient", nx=rng.randint(60, 140), ny=rng.randint(60, 130), nz=rng.randint(40, 72),
                    dtype=rng.choice(["float32", "float64"]), steps=rng.randint(60, 200), pml=rng.randint(6, 12),
                    checkpoint=rng.choice(["sqrt", "record"]))
    if kind == "complex":
        shape = tuple(rng.randint(40, 130) for _ in range(3))
        return grid_case(shape, rng.choice(["float64", "float32"]), rng.randint(10, 30), objects="complex",
                         pml=rng.randint(6, 10))
    low, high = {"small": (36, 80), "medium": (80, 200), "large": (200, 400)}[kind]
    shape = tuple(_log_int(rng, low, high) for _ in range(3))
    cells = shape[0] * shape[1] * shape[2]
    options = dict(pml=rng.randint(6, 16), material=rng.choice(["uniform", "noise", "spheres"]))
    if rng.random() < 0.5:
        options.update(objects=rng.choice(["plain", "absorbing"]), source=rng.choice(["point", "line", "plane"]),
                       detector=rng.choice(["none", "line", "block"]), material="uniform")
    if rng.random() < 0.15:
        options.update(periodic=True)
    return grid_case(shape, rng.choice(["float64", "float32", "float32", "float32c"]),
                     _steps(cells, 1.2e8, rng.randint(20, 60)), **options)


# ------------------------------------------------------------------ inputs
def _rng(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(1000003 * (int(seed) + 1))


def _smooth(gen, shape, cells=8):
    """Gaussian noise of correlation length ~`cells`, trilinearly interpolated."""
    coarse = torch.randn(tuple(n // cells + 2 for n in shape), generator=gen, device=DEV, dtype=torch.float32)
    return F.interpolate(coarse[None, None], size=shape, mode="trilinear", align_corners=True)[0, 0]


def _noise_eps(gen, shape):
    v = _smooth(gen, shape)
    return 1.0 + 11.0 * (v - v.min()) / (v.max() - v.min())


def _sphere_eps(gen, shape, count=24):
    """Dielectric spheres of 8-32 cells radius (an eighth of the edge at most)."""
    eps = torch.ones(shape, device=DEV, dtype=torch.float32)
    u = torch.rand((count, 5), generator=gen, device=DEV).cpu().tolist()
    ax = [torch.arange(n, device=DEV, dtype=torch.float32) for n in shape]
    rmax = max(4, min(32, min(shape) // 8))
    for cx, cy, cz, r, e in u:
        rad = rmax / 4 + r * rmax * 3 / 4
        d = ((ax[0] - cx * shape[0]) ** 2)[:, None, None] + ((ax[1] - cy * shape[1]) ** 2)[None, :, None] \
            + ((ax[2] - cz * shape[2]) ** 2)[None, None, :]
        eps[d <= rad * rad] = 1.0 + 11.0 * e
    return eps


def _grid_inputs(case, seed):
    """What a "grid" case is made of, as plain tensors and numbers."""
    shape = (case["nx"], case["ny"], case["nz"])
    gen = _rng(seed)
    flat = shape[2] == 1
    out = dict(shape=shape, courant=0.99 * (2 if flat else 3) ** -0.5)
    u = torch.rand(8, generator=gen, device=DEV).cpu().tolist()
    out["eps"] = {"uniform": lambda: 1.0, "noise": lambda: _noise_eps(gen, shape),
                  "spheres": lambda: _sphere_eps(gen, shape)}[case["material"]]()
    out["wave"] = dict(amplitude=0.5 + u[0], phase=6.0 * u[1], period=20 + int(20 * u[2]))
    # a source and a detector plane or line across the middle, objects between
    x0, y0, z0 = (int(0.30 * n) for n in shape)
    x1, y1, z1 = (max(int(0.70 * n), a + 1) for n, a in zip(shape, (x0, y0, z0)))
    xs, xd = int(0.25 * shape[0]), int(0.80 * shape[0])
    ym, zm = shape[1] // 2, shape[2] // 2
    out["source"] = {"point": (xs, ym, zm), "line": (xs, slice(y0, y1), zm),
                     "plane": (xs, slice(y0, y1), slice(z0, z1))}[case["source"]]
    # block detectors include the last index of each range
    out["detector"] = {"none": None, "line": (xd, slice(1, shape[1] - 1), zm),
                       "block": (slice(xd, xd), slice(y0, y1), slice(z0, z1))}[case["detector"]]
    objects = []
    if case["objects"] == "plain":
        objects.append(("plain", (slice(x0, x1), slice(y0, y1), slice(z0, z1)), dict(eps=2.0 + 2 * u[3])))
    elif case["objects"] == "complex":
        objects.append(("plain", (slice(x0, x1), slice(y0, y1), slice(z0, z1)),
                        dict(eps=complex(2.0 + 2 * u[3], 0.005 + 0.01 * u[4]))))
    elif case["objects"] == "absorbing":
        sx = max(2, round(24 * shape[0] / 512))
        xa = int(0.65 * shape[0])
        p = case["pml"]
        objects.append(("absorbing", (slice(xa, xa + sx), slice(p, shape[1] - p), slice(p, max(shape[2] - p, p + 1))),
                        dict(eps=2.0 + u[3], sigma=1e4)))
        box = tuple(max(2, n // 8) for n in shape)
        at = tuple(int(f * n) for f, n in zip((0.25, 0.40, 0.35), shape))
        q = torch.randn(box + (4,), generator=gen, device=DEV, dtype=torch.float64)
        lam = 1.0 + 8.0 * torch.rand(box + (3,), generator=gen, device=DEV, dtype=torch.float64)
        objects.append(("anisotropic", tuple(slice(a, a + n) for a, n in zip(at, box)), dict(inv=_spd_inverse(q, lam))))
    out["objects"] = objects
    out["E"] = torch.stack([0.1 * _smooth(gen, shape) for _ in range(3)], -1)
    out["H"] = torch.stack([0.1 * _smooth(gen, shape) for _ in range(3)], -1)
    return out


def _spd_inverse(q, lam):
    """R diag(1/lam) R^T per cell, R the rotation of the quaternion q."""
    q = q / q.norm(dim=-1, keepdim=True)
    w, x, y, z = q.unbind(-1)
    rows = [[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
            [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
            [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]]
    R = torch.stack([torch.stack(r, -1) for r in rows], -2)
    inv = torch.zeros_like(R)
    for a in range(3):
        for b in range(3):
            inv[..., a, b] = sum(R[..., a, k] * R[..., b, k] / lam[..., k] for k in range(3))
    return inv


def _faces(t, periodic):
    full = slice(None)
    keys = [(slice(0, t), full, full), (slice(-t, None), full, full), (full, slice(0, t), full),
            (full, slice(-t, None), full)]
    return keys if periodic else keys + [(full, full, slice(0, t)), (full, full, slice(-t, None))]


def _batch_inputs(case, seed):
    gen, out = _rng(seed), []
    n = case["count"]
    edges = torch.randint(case["low"], case["high"] + 1, (n, 3), generator=torch.Generator().manual_seed(17)).tolist()
    u = torch.rand((n, 5), generator=gen, device=DEV).cpu().tolist()
    for shape, w in zip(edges, u):
        p = case["pml"]
        at = tuple(p + int(f * (m - 2 * p)) for f, m in zip(w, shape))
        out.append(dict(shape=tuple(shape), courant=3 ** -0.5, eps=_noise_eps(gen, shape), source=at,
                        wave=dict(amplitude=0.5 + w[3], phase=6.0 * w[4], period=31), detector=None, objects=[],
                        E=torch.stack([0.1 * _smooth(gen, shape) for _ in range(3)], -1),
                        H=torch.stack([0.1 * _smooth(gen, shape) for _ in range(3)], -1)))
    return out


def _gradient_inputs(case, seed):
    gen = _rng(seed)
    shape = (case["nx"], case["ny"], case["nz"])
    nx, ny, nz = shape
    design = (slice(nx // 4, 3 * nx // 4), slice(ny // 4, 3 * ny // 4), slice(3 * nz // 8, 5 * nz // 8))
    size = tuple(s.stop - s.start for s in design)
    u = torch.rand(2, generator=gen, device=DEV).cpu().tolist()
    perm = 1.0 + 11.0 * torch.rand(size + (3,), generator=gen, device=DEV, dtype=torch.float64)
    p = case["pml"]
    return dict(shape=shape, courant=3 ** -0.5, eps=1.0, objects=[("plain", design, dict(eps=perm))], detector=None,
                source=(p + 4, slice(ny // 4, 3 * ny // 4), nz // 2),
                wave=dict(amplitude=0.5 + u[0], phase=6.0 * u[1], period=31),
                box=(nx - p - 6, slice(7 * ny // 16, 9 * ny // 16), slice(3 * nz // 8, 5 * nz // 8)))


# ------------------------------------------------------------ through fdtd
def _build(inputs, case, dtype):
    """The Grid of `inputs`, with its components, at its starting fields."""
    eps = inputs["eps"]
    grid = fdtd.Grid(inputs["shape"], grid_spacing=SPACING, courant_number=inputs["courant"],
                     permittivity=eps if not torch.is_tensor(eps) else eps[..., None])
    periodic = case.get("periodic", False)
    for key in _faces(case["pml"], periodic):
        grid[key] = fdtd.PML()
    if periodic:
        grid[:, :, 0] = fdtd.PeriodicBoundary()
    design = None
    for kind, key, par in inputs["objects"]:
        if kind == "plain":
            obj = fdtd.Object(permittivity=par["eps"])
        elif kind == "absorbing":
            obj = fdtd.AbsorbingObject(permittivity=par["eps"], conductivity=par["sigma"])
        else:
            obj = fdtd.AnisotropicObject(permittivity=1.0)
        grid[key] = obj
        if kind == "anisotropic":
            obj.inverse_permittivity = par["inv"].to(grid.obj_dtype)
        design = obj
    wave = inputs["wave"]
    args = dict(period=wave["period"], amplitude=wave["amplitude"], phase_shift=wave["phase"])
    slices = sum(isinstance(k, slice) for k in inputs["source"])
    grid[inputs["source"]] = (fdtd.PointSource, fdtd.LineSource, fdtd.PlaneSource)[slices](**args)
    detectors = []
    if inputs["detector"] is not None:
        block = isinstance(inputs["detector"][0], slice)
        detectors.append(fdtd.BlockDetector() if block else fdtd.LineDetector())
        grid[inputs["detector"]] = detectors[0]
    if "E" in inputs:
        grid.E = inputs["E"]
        grid.H = inputs["H"]
    return grid, detectors, design


def prepare(case, seed):
    fdtd.set_backend("hip." + case["dtype"])
    if case["kind"] == "batch":
        grids = [_build(i, case, case["dtype"])[0] for i in _batch_inputs(case, seed)]
        return dict(case=case, grids=grids, batch=GridBatch(grids))
    if case["kind"] == "gradient":
        inputs = _gradient_inputs(case, seed)
        grid, _, design = _build(inputs, case, case["dtype"])
        problem = IntensityGradient(grid, design, inputs["box"], case["steps"], case["checkpoint"])
        return dict(case=case, problem=problem, permittivity=inputs["objects"][0][2]["eps"])
    grid, detectors, _ = _build(_grid_inputs(case, seed), case, case["dtype"])
    return dict(case=case, grid=grid, detectors=detectors)


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        state["batch"].run(case["steps"])
        return dict(E=[g.E for g in state["grids"]], H=[g.H for g in state["grids"]])
    if case["kind"] == "gradient":
        objective, gradient = state["problem"].gradient(state["permittivity"])
        return dict(objective=objective, gradient=gradient)
    grid = state["grid"]
    if case["call"] == "step":
        for _ in range(case["steps"]):
            grid.step()
    else:
        grid.run(case["steps"], progress_bar=False)
    return dict(E=grid.E, H=grid.H, E_read=[d.trace("E") for d in state["detectors"]],
                H_read=[d.trace("H") for d in state["detectors"]])


# -------------------------------------------------------------------- work
def _step_work(shape, pml, periodic, dtype, is_complex=False):
    """Bytes and operations of one step: E, H and both materials read once, E
    and H written once, two CPML values per field, face and slab cell read and
    written once; 21 operations per cell and half step, 9 per face cell."""
    nx, ny, nz = shape
    cells = nx * ny * nz
    slab = 2 * pml * (ny * nz + nx * nz) + (0 if periodic else 2 * pml * nx * ny)
    value = ITEM[dtype] * (2 if is_complex else 1)
    psi = (8 if dtype == "float32c" else ITEM[dtype]) * (2 if is_complex else 1)
    material = 2 if dtype == "float32c" else 6 * ITEM[dtype]
    k = 2 if is_complex else 1
    return cells * (12 * value + material) + slab * 8 * psi, (42 * cells + 18 * slab) * k


def work(case):
    if case["kind"] == "batch":
        per = [_step_work(i, case["pml"], False, case["dtype"]) for i in _batch_shapes(case)]
        return {"bytes": case["steps"] * sum(b for b, _ in per), "flops": case["steps"] * sum(f for _, f in per)}
    shape = (case["nx"], case["ny"], case["nz"])
    b, f = _step_work(shape, case["pml"], case.get("periodic", False), case["dtype"],
                      case.get("objects") == "complex")
    # a gradient takes each step forward and its transpose back
    k = case["steps"] * (2 if case["kind"] == "gradient" else 1)
    return {"bytes": b * k, "flops": f * k}


def _batch_shapes(case):
    gen = torch.Generator().manual_seed(17)
    return torch.randint(case["low"], case["high"] + 1, (case["count"], 3), generator=gen).tolist()


# ------------------------------------------------- the same in plain float64
class _Plain:
    """One grid stepped in 64 bits with array operations (out of place, so
    that it can be differentiated)."""

    def __init__(self, inputs, case):
        self.inputs, self.case = inputs, case
        shape, S = inputs["shape"], inputs["courant"]
        self.S = S
        self.wide = torch.complex128 if case.get("objects") == "complex" else torch.float64
        eps = inputs["eps"]
        # a single-precision backend is given its permittivity in that type
        eps = eps.double() if torch.is_tensor(eps) else torch.full(shape, float(eps), device=DEV, dtype=torch.float64)
        self.K = torch.stack([S / eps] * 3)
        self.objects = []
        last = self.K / S
        for kind, key, par in inputs["objects"]:
            size = tuple(s.stop - s.start for s in key)
            if kind == "anisotropic":
                inv = par["inv"]
            else:
                inv = self.inverse(par["eps"], size, key, last)
            self.objects.append((kind, key, inv, par))
            last[(slice(None),) + key] = 0
        self.K = last * S
        self.profiles()
        like = dict(device=DEV, dtype=self.wide)
        self.E = inputs["E"].permute(3, 0, 1, 2).to(self.wide) if "E" in inputs else torch.zeros((3,) + shape, **like)
        self.H = inputs["H"].permute(3, 0, 1, 2).to(self.wide) if "H" in inputs else torch.zeros((3,) + shape, **like)
        zero = torch.zeros((), **like)
        # psi[axis][component differenced], full size where the axis has faces
        self.psiE = [[zero.expand(shape)] * 2 if self.cE[a] is not None else None for a in range(3)]
        self.psiH = [[zero.expand(shape)] * 2 if self.cE[a] is not None else None for a in range(3)]
        self.E_read, self.H_read = [], []

    def inverse(self, eps, size, key, last):
        """1/eps of an object; its last plane along each axis takes the grid's
        value from the grid's last plane for the component normal to it."""
        if not torch.is_tensor(eps):
            eps = torch.full(size + (3,), eps, device=DEV, dtype=self.wide)
        inv = (1.0 / eps).permute(3, 0, 1, 2)
        for c in range(3):
            if size[c] > 1:
                src = list(key)
                src[c] = slice(-1, None)
                mask = torch.zeros(size[c], dtype=torch.bool, device=DEV)
                mask[-1] = True
                mask = mask.view([-1 if a == c else 1 for a in range(3)]).expand(size)
                edge = last[(c,) + tuple(src)].to(inv.dtype).expand(size)
                inv = torch.stack([torch.where(mask, edge, inv[d]) if d == c else inv[d] for d in range(3)])
        return inv

    def profiles(self):
        """CPML decay b and gain c along each axis, for E and H."""
        shape, t, a = self.inputs["shape"], self.case["pml"], 1e-8
        self.bE, self.cE, self.bH, self.cH = ([None] * 3 for _ in range(4))
        for ax in range(3):
            if ax == 2 and self.case.get("periodic", False):
                continue
            n = shape[ax]
            sig = lambda v: 40 * v ** 3 / (t + 1) ** 4
            up = torch.arange(t, device=DEV, dtype=torch.float64)
            sE = torch.zeros(n, device=DEV, dtype=torch.float64)
            sH = torch.zeros_like(sE)
            gE, gH = torch.zeros_like(sE), torch.zeros_like(sE)
            sE[:t], sE[n - t:] = sig(t - 0.5 - up), sig(up + 0.5)
            sH[:t - 1], sH[n - t:n - 1] = sig(t - 1 - up[:t - 1]), sig(up[1:])
            gE[1:t], gE[n - t + 1:] = 1, 1
            gH[:t - 1], gH[n - t:n - 1] = 1, 1
            view = [-1 if d == ax else 1 for d in range(3)]
            for s, g, b_, c_ in ((sE, gE, self.bE, self.cE), (sH, gH, self.bH, self.cH)):
                b = torch.exp(-(s + a) * self.S)
                b_[ax] = b.view(view)
                c_[ax] = ((b - 1) * s / (s + a) * g).view(view)

    @staticmethod
    def diff(f, axis, back):
        n = f.shape[axis]
        d = f.narrow(axis, 1, n - 1) - f.narrow(axis, 0, n - 1)
        pad = [0, 0] * (2 - axis) + ([1, 0] if back else [0, 1])
        return F.pad(d, pad)

    def curl(self, f, psi, b, c, back):
        """(curl, CPML term) of the field f; psi is updated."""
        out = [None] * 3
        phi = [None] * 3
        for k in range(3):
            p, q = (k + 1) % 3, (k + 2) % 3  # + d f_q / d p - d f_p / d q
            dq, dp = self.diff(f[q], p, back), self.diff(f[p], q, back)
            out[k] = dq - dp
            for ax, d, sign, slot in ((p, dq, 1, 0), (q, dp, -1, 1)):
                if psi[ax] is None:
                    continue
                new = list(psi[ax])
                new[slot] = psi[ax][slot] * b[ax] + d * c[ax]
                psi[ax] = new
                phi[k] = (phi[k] if phi[k] is not None else 0) + sign * new[slot]
            if phi[k] is None:
                phi[k] = torch.zeros_like(out[k])
        return out, phi

    def wave(self, q):
        w = self.inputs["wave"]
        return math.sin(2 * math.pi * q / w["period"] + w["phase"]) * w["amplitude"]

    def sources(self, f, q, is_H):
        key = self.inputs["source"]
        slices = sum(isinstance(k, slice) for k in key)
        if slices == 2:  # a hard plane source normal to x sets E_z and H_y
            f = f.clone()
            f[(1 if is_H else 2,) + key] = self.wave(q)
            return f
        if is_H:
            return f
        value = self.wave(q)
        if slices == 1:
            n = key[1].stop - key[1].start
            d2 = (torch.arange(n, device=DEV, dtype=torch.float64) - n // 2) ** 2
            prof = torch.exp(-(d2 ** 2) / (2 * (0.5 * d2.max()) ** 2))
            value = value * prof / prof.sum()
        add = torch.zeros(self.inputs["shape"], device=DEV, dtype=f.dtype)
        add[key] = value
        return torch.stack([f[0], f[1], f[2] + add])

    def sample(self, f, into):
        key = self.inputs["detector"]
        if key is None:
            return
        if isinstance(key[0], slice):
            key = tuple(slice(k.start, k.stop + 1) for k in key)
        into.append(f[(slice(None),) + key].movedim(0, -1).clone())

    def step(self, q):
        S = self.S
        curl, phi = self.curl(self.H, self.psiE, self.bE, self.cE, True)
        E = torch.stack([self.E[c] + self.K[c] * curl[c] for c in range(3)])
        for kind, key, inv, par in self.objects:
            box = (slice(None),) + key
            cu = torch.stack([c[key] for c in curl])
            if kind == "plain":
                new = E[box] + S * inv * cu
            elif kind == "absorbing":
                f = 0.5 * S * inv * par["sigma"] * SPACING * 4e-7 * math.pi * C0
                new = E[box] * ((1 - f) / (1 + f)) + S * inv * cu / (1 + f)
            else:
                new = E[box] + S * torch.stack([sum(inv[..., r, c] * cu[c] for c in range(3)) for r in range(3)])
            E = E.clone()
            E[box] = new
        E = torch.stack([E[c] + self.K[c] * phi[c] for c in range(3)])
        if self.case.get("periodic", False) and E.shape[3] > 1:
            E = torch.cat([E[..., -1:], E[..., 1:]], 3)
        self.E = self.sources(E, q, False)
        self.sample(self.E, self.E_read)
        curl, phi = self.curl(self.E, self.psiH, self.bH, self.cH, False)
        H = torch.stack([self.H[c] - S * (curl[c] + phi[c]) for c in range(3)])
        if self.case.get("periodic", False) and H.shape[3] > 1:
            H = torch.cat([H[..., :-1], H[..., :1]], 3)
        self.H = self.sources(H, q, True)
        self.sample(self.H, self.H_read)

    def state(self):
        return [self.E, self.H] + [t for p in self.psiE + self.psiH if p is not None for t in p]

    def load(self, state):
        self.E, self.H, rest = state[0], state[1], list(state[2:])
        for p in (self.psiE, self.psiH):
            for a in range(3):
                if p[a] is not None:
                    p[a] = [rest.pop(0), rest.pop(0)]


def _exact_gradient(case, seed):
    from torch.utils.checkpoint import checkpoint

    inputs = _gradient_inputs(case, seed)
    kind, key, par = inputs["objects"][0]
    perm = par["eps"].clone().requires_grad_(True)
    inputs["objects"] = [(kind, key, dict(eps=perm))]
    sim = _Plain(inputs, case)
    box = (slice(None),) + inputs["box"]
    seg = max(1, math.isqrt(case["steps"]))
    inv = sim.objects[0][2]

    def segment(q0, q1, inv_, *state):
        sim.load(state)
        sim.objects[0] = (kind, key, inv_, par)
        J = 0
        for q in range(q0, q1):
            sim.step(q)
            J = J + sim.E[box].square().sum()
        return (J,) + tuple(sim.state())

    total, state = 0, sim.state()
    for q0 in range(0, case["steps"], seg):
        J, *state = checkpoint(segment, q0, min(q0 + seg, case["steps"]), inv, *state, use_reentrant=False)
        total = total + J
    total.backward()
    return dict(objective=float(total.detach()), gradient=perm.grad)


def exact(case, seed):
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    with torch.no_grad():
        if case["kind"] == "batch":
            out = dict(E=[], H=[])
            for inputs in _batch_inputs(case, seed):
                sim = _Plain(inputs, case)
                for q in range(case["steps"]):
                    sim.step(q)
                out["E"].append(sim.E.movedim(0, -1))
                out["H"].append(sim.H.movedim(0, -1))
            return out
        sim = _Plain(_grid_inputs(case, seed), case)
        for q in range(case["steps"]):
            sim.step(q)
        read = [[torch.stack(r)] if r else [] for r in (sim.E_read, sim.H_read)]
        return dict(E=sim.E.movedim(0, -1), H=sim.H.movedim(0, -1), E_read=read[0], H_read=read[1])
