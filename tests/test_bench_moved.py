"""The bytes a step is credited with are those its kernels move (CPU only)."""
import importlib.util
import os

import pytest

from distributednavierstokes_amd.workloads import channel_problem

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_shared_passes_are_not_counted(bench):
    prob = channel_problem((256, 192, 256), "explicit", "fp64")
    model = bench.mmin_units_per_step(prob)
    assert bench.moved_units_per_step(prob, {"stages": "separate", "cn": "seg3"}) == model
    moved = bench.moved_units_per_step(prob, {"stages": "fused zc=16"})
    # the momentum launches of the two forms differ by the same amount as the steps, less the two gradient passes
    a, b = (3 * bench.family_bytes_per_launch(prob, 0, 8, fused=f) / (256 * 192 * 256 * 8) for f in (False, True))
    assert abs(model - moved - (2 * 7 - (b - a))) < 1e-9 and moved == model - 12


def test_pressure_rows_read_once(bench):
    prob = channel_problem((512, 384, 512), "implicit", "fp64")
    model = bench.mmin_units_per_step(prob)
    assert bench.moved_units_per_step(prob, {"stages": "separate", "cn": "seg R=24"}) == model
    one, three = (bench.family_bytes_per_launch(prob, 5, 8, cn3=c) / (512 * 384 * 512 * 8) for c in (False, True))
    assert model - bench.moved_units_per_step(prob, {"cn": "seg3 R=24 p=lds"}) == 3 * (3 * one - three)
    plain = channel_problem((512, 384, 512), "implicit", "plain")
    assert bench.moved_units_per_step(plain, {"stages": "fused", "cn": "seg3"}) == bench.mmin_units_per_step(plain)
