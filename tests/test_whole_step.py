"""Whole steps (one kernel a step) against half steps, and the main form of the
half-step kernels against the general one, bit for bit: the forms of
tests/step_forms.py on the CPU build of the kernels (under AddressSanitizer)
and on the GPU, and the size rule of the whole steps on the GPU."""

import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests"))

import step_forms  # noqa: E402


def run_on_the_host(forms, *options):
    sys.path.insert(0, os.path.join(ROOT, "tests", "cpu_kernels"))
    import build

    build.build()
    env = dict(os.environ, LD_PRELOAD=build.asan_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    child = os.path.join(ROOT, "tests", "cpu_kernels", "step_forms_child.py")
    res = subprocess.run([sys.executable, child, *options] + forms, capture_output=True, text=True, env=env, timeout=600)
    lines = [json.loads(x) for x in res.stdout.splitlines() if x.startswith("{")]
    assert res.returncode == 0, res.stderr[-4000:]
    assert [r["form"] for r in lines] == forms
    assert not [r for r in lines if r["bad"]]


def backends(name):
    return step_forms.BACKENDS[:2] if name == "complex" else step_forms.BACKENDS


def test_whole_steps_on_the_host():
    run_on_the_host([f"{n}/hip.float64" for n in step_forms.FORMS]
                    + [f"{n}/{b}" for n in ("plane", "detectors", "five_points", "objects")
                       for b in step_forms.BACKENDS[1:]])


def test_main_form_on_the_host():
    run_on_the_host([f"{n}/hip.float64" for n in ("one_cell_rows", "flat_x", "cube", "z_first", "slabs_meet", "objects",
                                                  "five_points", "many_tiles", "complex")]
                    + [f"{n}/{b}" for n in ("flat_z", "objects") for b in step_forms.BACKENDS[1:]], "--half")


def test_transposed_forms_on_the_host():
    run_on_the_host([f"{n}/{b}" for n in step_forms.GRADIENTS for b in step_forms.BACKENDS[:2]], "--gradient")


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(step_forms.GRADIENTS))
@pytest.mark.parametrize("backend", step_forms.BACKENDS[:2])
def test_transposed_forms_match(name, backend):
    import fdtd_amd as fdtd

    assert step_forms.gradient_differences(fdtd, name, backend) == []


@pytest.mark.gpu
@pytest.mark.parametrize("name,backend", [(n, b) for n in step_forms.FORMS for b in backends(n)])
def test_whole_steps_match_half_steps(name, backend):
    import fdtd_amd as fdtd

    assert step_forms.differences(fdtd, name, backend) == []


@pytest.mark.gpu
@pytest.mark.parametrize("name,backend", [(n, b) for n in step_forms.FORMS for b in backends(n)])
def test_main_form_matches_general_form(name, backend):
    import fdtd_amd as fdtd

    assert step_forms.form_differences(fdtd, name, backend) == []


@pytest.mark.gpu
@pytest.mark.parametrize("shape,backend,taken", [((64, 64, 64), "hip.float64", True), ((64, 64, 64), "hip.float32", True),
                                                 ((65, 64, 64), "hip.float32", False), ((1100, 1000, 1), "hip.float64", False), ((128, 96, 96), "hip.float64", False),
                                                 ((1000, 700, 1), "hip.float32", True)])
def test_size_rule(shape, backend, taken):
    import fdtd_amd as fdtd

    fdtd.set_backend(backend)
    grid = fdtd.Grid(shape, grid_spacing=100e-9)
    grid[0:6] = fdtd.PML()
    grid.run(2, progress_bar=False)
    assert step_forms.whole(grid) == taken
