"""Whole steps (one kernel a step) against half steps, bit for bit: the forms
of tests/step_forms.py on the CPU build of the kernels (under
AddressSanitizer) and on the GPU, and the size rule on the GPU."""

import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests"))

import step_forms  # noqa: E402


def test_whole_steps_on_the_host():
    sys.path.insert(0, os.path.join(ROOT, "tests", "cpu_kernels"))
    import build

    lib, asan = build.build(), build.asan_runtime()
    env = dict(os.environ, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    forms = [f"{n}/hip.float64" for n in step_forms.FORMS]
    forms += [f"{n}/{b}" for n in ("plane", "detectors", "five_points", "objects") for b in step_forms.BACKENDS[1:]]
    res = subprocess.run([sys.executable, os.path.join(ROOT, "tests", "cpu_kernels", "step_forms_child.py")] + forms,
                         capture_output=True, text=True, env=env, timeout=600)
    lines = [json.loads(x) for x in res.stdout.splitlines() if x.startswith("{")]
    assert res.returncode == 0, res.stderr[-4000:]
    assert [r["form"] for r in lines] == forms
    assert not [r for r in lines if r["bad"]]


@pytest.mark.gpu
@pytest.mark.parametrize("backend", step_forms.BACKENDS)
@pytest.mark.parametrize("name", list(step_forms.FORMS))
def test_whole_steps_match_half_steps(name, backend):
    import fdtd_amd as fdtd

    assert step_forms.differences(fdtd, name, backend) == []


@pytest.mark.gpu
@pytest.mark.parametrize("shape,backend,taken", [((64, 64, 64), "hip.float64", True), ((64, 64, 64), "hip.float32", False),
                                                 ((50, 51, 50), "hip.float32", True), ((128, 96, 96), "hip.float64", False),
                                                 ((1000, 700, 1), "hip.float32", True)])
def test_size_rule(shape, backend, taken):
    import fdtd_amd as fdtd

    fdtd.set_backend(backend)
    grid = fdtd.Grid(shape, grid_spacing=100e-9)
    grid[0:6] = fdtd.PML()
    grid.run(2, progress_bar=False)
    assert step_forms.whole(grid) == taken
