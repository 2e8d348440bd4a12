"""cyr_set_energy_lanes where the E-basis runs separate Y and z passes (FP64 in 3D, columns
without a codelet)."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from tests.helpers import random_constants, random_euler

torch = pytest.importorskip("torch")

GRIDS = [((40, 36, 12), capi.FP64), ((64, 64, 32), capi.FP64), ((48, 50, 20), capi.FP32), ((60, 90, 1), capi.FP32)]


@pytest.fixture
def lanes():
    before = capi.energy_lanes()
    yield capi.set_energy_lanes
    capi.set_energy_lanes(before)


def _sim(dims, prec, frame=1):
    return capi.Sim(dims, 2, 2.0, [283.0, 285.0, 286.0, 288.0, 290.0], (0, 15, 165), precision=prec,
                    pipeline=capi.PIPE_EBASIS, interpolation=1, windowing=1, reference_frame=frame)


@pytest.mark.parametrize("dims,prec", GRIDS)
def test_two_lanes_hold_two_units(dims, prec, lanes):
    sim, V = _sim(dims, prec), dims[0] * dims[1] * dims[2]
    lanes(1)
    one = sim.footprint()
    lanes(2)
    assert sim.footprint() - one >= 5 * V * (16 if prec == capi.FP64 else 8)


@pytest.mark.gpu
@pytest.mark.parametrize("frame", [1, 0])
@pytest.mark.parametrize("dims,prec", GRIDS)
def test_two_lanes_bitwise(dims, prec, frame, lanes):
    print(f"two lanes {dims} prec={prec} frame={frame}", flush=True)
    sim = _sim(dims, prec, frame)
    vox, mats = random_euler(dims, 2, 51), random_constants(5, 2, 52)
    lanes(1)
    ref = capi.simulate(sim, vox, mats)
    lanes(2)
    for _ in range(3):
        np.testing.assert_array_equal(capi.simulate(sim, vox, mats), ref)
