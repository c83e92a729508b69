"""Grids whose ``run`` may take whole steps (one kernel a step), and a
comparison of such a run with the same run taken half step by half step
(FDTD_HIP_STEP=0): every field, CPML and trace value must have the same bits.

The forms cover the whole-step rule and its edges: flat and 3D grids smaller
than a tile, of one cell more than a tile, and of many tiles with remainders;
CPML on any side, of any thickness, in any registration order (orders that
differ between sides, and slabs that overlap, go half by half); every object
kind; folded and unfolded point sources, straight, diagonal and list lines,
plane sources; line, diagonal and block detectors (sources or detectors that
name a cell twice go half by half).
"""

import os

import numpy as np
import torch

S = slice
FULL = (S(None), S(None), S(None))


def face(axis, high, t):
    key = list(FULL)
    key[axis] = S(-t, None) if high else S(0, t)
    return ("PML", {}, tuple(key))


def faces(t, axes=(0, 1, 2)):
    return [face(a, h, t) for a in axes for h in (0, 1)]


POINT = ("PointSource", dict(period=9, amplitude=0.7), "mid")
FORMS = {
    # name: (shape, components, whether whole steps are taken)
    "one_cell_rows": ((37, 1, 1), [face(0, 0, 4), face(0, 1, 3), POINT], True),
    "flat_z": ((23, 41, 1), faces(5, (0, 1)) + [("PeriodicBoundary", {}, (S(None), S(None), 0)), POINT], True),
    "flat_x": ((1, 19, 30), faces(4, (1, 2)) + [POINT], True),
    "flat_y": ((33, 1, 18), faces(3, (2, 0)) + [POINT], True),
    "cube": ((17, 18, 19), faces(4) + [POINT], True),
    "no_faces": ((9, 7, 5), [POINT], True),
    "thin_faces": ((11, 10, 23), faces(1) + [POINT], True),
    "one_side": ((14, 13, 12), [face(1, 1, 5), face(2, 0, 6), POINT], True),
    "z_first": ((13, 12, 15), faces(3, (2, 0, 1)) + [POINT], True),
    "mixed_order": ((13, 12, 15), [face(0, 0, 3), face(1, 1, 3), face(0, 1, 3), face(1, 0, 3), POINT], False),
    "overlapping_slabs": ((7, 12, 11), [face(0, 0, 5), face(0, 1, 5), POINT], False),
    "periodic": ((10, 11, 12), faces(3, (0, 1)) + [("PeriodicBoundary", {}, (S(None), S(None), 0)), POINT], False),
    "slabs_meet": ((8, 12, 11), [face(0, 0, 4), face(0, 1, 4), POINT], True),
    "objects": ((18, 17, 16), faces(3) + [
        ("Object", dict(permittivity=2.5), (S(4, 9), S(3, 8), S(5, 12))),
        ("AbsorbingObject", dict(permittivity=1.5, conductivity=2e4), (S(8, 13), S(6, 11), S(2, 9))),
        ("AnisotropicObject", dict(permittivity=2.0), (S(11, 15), S(9, 14), S(10, 13))), POINT], True),
    "five_points": ((15, 14, 13), faces(3) + [("PointSource", dict(period=7 + n), (3 + n, 4 + n, 5)) for n in range(5)]
                    + [("PointSource", dict(period=8), (3, 4, 5))], True),
    "lines": ((20, 17, 15), faces(3) + [
        ("LineSource", dict(period=11), (4, S(3, 12), 7)),
        ("LineSource", dict(period=12), (S(5, 15), S(2, 9), 9)),
        ("LineSource", dict(period=13), ([9, 5, 12], [8, 8, 3], [4, 4, 10]))], True),
    "repeated_cell": ((14, 13, 12), faces(3) + [
        POINT, ("LineDetector", {}, ([4, 5, 4], [6, 6, 6], [7, 7, 7]))], False),
    "plane": ((14, 19, 17), faces(3) + [
        ("PlaneSource", dict(period=15, polarization="y"), (5, S(4, 15), S(3, 12))),
        ("LineSource", dict(period=11), (5, S(3, 12), 7))], True),
    "detectors": ((17, 15, 14), faces(3) + [
        ("LineDetector", {}, (S(2, 14), 7, 6)), ("LineDetector", {}, (S(3, 13), S(2, 12), S(1, 11))),
        ("BlockDetector", {}, (S(4, 7), S(9, 9), S(2, 11))), POINT], True),
    # lists that the half steps' tail spreads over workgroups: in one launch,
    # the reads in a launch of their own, sources that share cells
    "wide_apart": ((6, 48, 41), faces(2, (1, 2)) + [
        ("PlaneSource", dict(period=15, polarization="z"), (2, S(1, 46), S(1, 40))),
        ("BlockDetector", {}, (S(4, 4), S(1, 45), S(1, 38)))], True),
    "wide_read_sources": ((6, 48, 41), faces(2, (1, 2)) + [
        ("PlaneSource", dict(period=15, polarization="y"), (2, S(1, 46), S(1, 40))),
        ("LineSource", dict(period=11), (4, S(3, 42), 7)),
        ("BlockDetector", {}, (S(2, 4), S(1, 45), S(1, 38)))], True),
    "wide_shared": ((6, 48, 41), faces(2, (1, 2)) + [
        ("PlaneSource", dict(period=15, polarization="y"), (2, S(1, 46), S(1, 40))),
        ("PlaneSource", dict(period=13, polarization="x"), (S(1, 5), 20, S(1, 40))),
        ("LineSource", dict(period=11), (2, S(3, 42), 7)),
        ("BlockDetector", {}, (S(1, 4), S(1, 45), S(1, 38)))], True),
    "many_tiles": ((21, 34, 67), faces(6) + [POINT], True),
    "complex": ((12, 19, 17), faces(3) + [
        ("Object", dict(permittivity=2.5 + 0.03j), (S(3, 8), S(3, 9), S(5, 12))),
        ("AbsorbingObject", dict(permittivity=1.5, conductivity=2e4), (S(7, 10), S(6, 11), S(2, 9))), POINT], False),
}
BACKENDS = ("hip.float64", "hip.float32", "hip.float32c")
RUNS = (4, 1, 3)  # even, single and odd runs, half steps and an edit between them


def build(fdtd, name, seed=0):
    shape, comps, _ = FORMS[name]
    rng = np.random.RandomState(seed)
    eps = rng.uniform(1.0, 4.0, size=shape + (3,))
    mu = rng.uniform(1.0, 2.0, size=shape + (3,))
    grid = fdtd.Grid(shape, grid_spacing=100e-9, courant_number=0.5, permittivity=torch.from_numpy(eps),
                     permeability=torch.from_numpy(mu))
    for kind, params, key in comps:
        if key == "mid":
            key = tuple(n // 2 for n in shape)
        grid[key] = getattr(fdtd, kind)(**params)
    grid.E = torch.from_numpy(0.1 * rng.randn(*shape, 3))
    grid.H = torch.from_numpy(0.1 * rng.randn(*shape, 3))
    return grid


def state(grid):
    out = [grid._E_rec, grid._H_rec] if grid.compensated else [grid._E, grid._H]
    for b in grid.boundaries:
        out += [t for t in (getattr(b, "_psiE", None), getattr(b, "_psiH", None)) if t is not None]
    for d in grid.detectors:
        out += [d.trace("E"), d.trace("H")]
    return [t.clone() for t in out]


def advance(grid):
    """RUNS with a state after each, half steps and a material edit between."""
    out = []
    for n in RUNS:
        grid.run(n, progress_bar=False)
        out += state(grid)
        grid.update_E()
        grid.update_H()
        grid.time_steps_passed += 1
        grid.inverse_permittivity[0] *= 0.5
    return out


def traced(fdtd, name, backend, env):
    """The states of `advance` under the environment `env`, and the grid."""
    fdtd.set_backend(backend)
    keep = dict(os.environ)
    try:
        os.environ.update(env)
        grid = build(fdtd, name)
        return advance(grid), grid
    finally:
        os.environ.clear()
        os.environ.update(keep)


def unequal(got, want):
    return [f"state {i}" for i, (a, b) in enumerate(zip(got, want))
            if not torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))]


# launches of the half steps: x planes a workgroup, tile shape, objects in a
# launch of their own
SHAPES = {f"cx{cx}_{tile}_{objs}": {"FDTD_HIP_STEP": "0", "FDTD_HIP_CX": str(cx), "FDTD_HIP_FLAT": flat,
                                    "FDTD_HIP_OBJECT_TILES": tiles}
          for cx in (1, 2, 3) for tile, flat in (("flat", "1"), ("rows", "0"))
          for objs, tiles in (("joint", "0"), ("apart", "1"))}


def form_differences(fdtd, name, backend, shapes=tuple(SHAPES)):
    """Launch shapes at which the main form of the half-step kernels differs
    from the general one."""
    want, _ = traced(fdtd, name, backend, {"FDTD_HIP_STEP": "0", "FDTD_HIP_GENERAL": "1"})
    bad = []
    for shape in shapes:
        got, _ = traced(fdtd, name, backend, SHAPES[shape])
        bad += [f"{shape}: {d}" for d in unequal(got, want)]
    return bad


def whole(grid):
    """Whether the grid's plan took whole steps."""
    return isinstance(grid._plan.step_buf, torch.Tensor)


def differences(fdtd, name, backend):
    """Names of what is wrong: differing states, or the other route taken."""
    want, half = traced(fdtd, name, backend, {"FDTD_HIP_STEP": "0"})
    got, grid = traced(fdtd, name, backend, {"FDTD_HIP_STEP": "1"})
    bad = unequal(got, want)
    if whole(half):
        bad.append("half steps were asked for")
    if whole(grid) != FORMS[name][2]:
        bad.append(f"whole steps: {whole(grid)}")
    return bad


# Gradients: the transposed half steps' form for slabs that do not overlap
# against their general form (FDTD_HIP_ADJ_FULL=0), and the field recorded by
# the E kernel (up to 4 point sources) against the record of the tail (5).
GRADIENTS = {
    # name: (shape, CPML thickness, axes with faces, further objects)
    "cube": ((17, 18, 19), 4, (0, 1, 2), []),
    "long_rows": ((9, 7, 71), 2, (0, 1, 2), []),
    "slabs_meet": ((8, 12, 14), 4, (0, 1, 2), []),
    "thin_faces": ((11, 10, 23), 1, (0, 1, 2), []),
    "no_faces": ((9, 8, 7), 0, (), []),
    "one_axis": ((10, 16, 33), 5, (2,), []),
    "absorber": ((17, 16, 15), 3, (0, 1, 2), [("AbsorbingObject", dict(permittivity=2.0, conductivity=1e4),
                                               (S(11, 14), S(3, 12), S(4, 11)))]),
    "anisotropic": ((17, 16, 15), 3, (1, 2), [("AnisotropicObject", dict(permittivity=2.0),
                                               (S(11, 14), S(3, 12), S(4, 11)))]),
}
ADJOINT_SHAPES = [{"FDTD_HIP_ADJ_CX": str(cx), "FDTD_HIP_FLAT": flat} for cx in (1, 2, 3) for flat in ("1", "0")]


def gradient(fdtd, name, sources):
    from fdtd_amd.adjoint import IntensityGradient

    shape, t, axes, objects = GRADIENTS[name]
    rng = np.random.RandomState(3)
    grid = fdtd.Grid(shape, grid_spacing=100e-9, courant_number=0.5,
                     permittivity=torch.from_numpy(rng.uniform(1.0, 3.0, size=shape + (3,))))
    for kind, params, key in faces(t, axes) if t else []:
        grid[key] = fdtd.PML()
    mid = [n // 2 for n in shape]
    grid[tuple(mid)] = fdtd.PointSource(period=9, amplitude=0.7)
    for _ in range(sources - 1):
        grid[tuple(mid)] = fdtd.PointSource(period=9, amplitude=0.0)
    box = (S(mid[0] - 3, mid[0] + 1), S(mid[1] - 3, mid[1] + 3), S(mid[2] - 2, mid[2] + 3))
    perm = torch.from_numpy(rng.uniform(1.0, 3.0, size=(4, 6, 5, 3)))
    design = fdtd.Object(perm, name="design")
    grid[box] = design
    for kind, params, key in objects:
        grid[key] = getattr(fdtd, kind)(**params)
    prob = IntensityGradient(grid, design, (mid[0] + 1, S(1, shape[1] - 1), S(2, shape[2] - 1)), 12, checkpoint="record")
    J, g = prob.gradient(perm)
    return J, g.clone()


def gradient_differences(fdtd, name, backend):
    fdtd.set_backend(backend)
    keep = dict(os.environ)
    out = []
    try:
        os.environ.update(ADJOINT_SHAPES[0], FDTD_HIP_ADJ_FULL="0")
        J, g = gradient(fdtd, name, 5)
        if not bool(torch.isfinite(g).all()) or float(g.abs().max()) == 0.0:
            return ["gradient not finite or all zero"]
        os.environ["FDTD_HIP_ADJ_FULL"] = "1"
        for env in ADJOINT_SHAPES:
            os.environ.update(env)
            J1, g1 = gradient(fdtd, name, 1)
            if J1 != J or not torch.equal(g, g1):
                out.append(f"{env}: J {J!r} against {J1!r}, gradient {float((g - g1).abs().max())!r} apart")
    finally:
        os.environ.clear()
        os.environ.update(keep)
    return out
