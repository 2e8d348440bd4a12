"""The rotation of small planes (angles split over the waves of a block, 4 or 16) and the
quarter-turn orbits (one orbit pixel per wave) against the oracle, and the E-basis
executor's quadratic forms that feed them.  Sizes around the rules' edges: planes of
one tile, ragged tiles, fewer angles than waves, enough energies or pixels for the
one-wave-per-quadrant kernels.  Bars: FP64 1e-10, FP32 1e-4, identical masks."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")

CASES = {
    # (dims, energies, angles, options)
    "one_angle": ((16, 16, 4), 1, (0.0, 1.0, 0.0), {}),
    "few_angles_ragged": ((45, 37, 4), 2, (0.0, 50.0, 100.0), dict(rot_mask=1)),
    "sixteen_waves": ((40, 40, 6), 1, (0.0, 10.0, 170.0), {}),
    "four_waves": ((96, 80, 2), 8, (0.0, 12.0, 168.0), dict(rot_mask=1)),
    "orbits_half_turn": ((128, 128, 1), 33, (0.0, 15.0, 165.0), dict(rot_mask=1)),
    "orbits_full_turn": ((128, 128, 1), 34, (0.0, 30.0, 330.0), {}),
    "orbits_three_quarters": ((130, 130, 1), 34, (0.0, 30.0, 240.0), {}),
    "general_many_energies": ((120, 128, 1), 34, (0.0, 15.0, 165.0), {}),
}


@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("case", sorted(CASES))
def test_rotation_routes(case, prec):
    dims, nE, angles, kw = CASES[case]
    print(f"rotation {case} prec={prec}", flush=True)
    vox = random_euler(dims, 2, 12)
    energies = list(280.0 + 0.25 * np.arange(nE))
    mats = random_constants(nE, 2, 13)
    kw = dict(kw, interpolation=1)
    phys = 2.0 if dims[2] == 1 else 5.0
    ref = O.simulate(O.Sim(dims, 2, phys, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, 2, phys, energies, angles, precision=prec, pipeline=pipeline, **kw)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        print(f"  pipeline {pipeline}: rel L2 {err:.3e}")
        assert same, (case, pipeline)
        assert err < (1e-10 if prec == capi.FP64 else 1e-4), (case, pipeline, err)


def test_tilted_beam_radius():
    """E-basis rotation with the Ewald disc off the plane's centre: tiles beyond the disc's
    farthest point are filled, none inside it."""
    dims, energies, angles = (64, 48, 8), [285.0], (0.0, 30.0, 150.0)
    vox, mats = random_euler(dims, 2, 8), random_constants(1, 2, 9)
    k = np.array([[0.0, 0.3, 1.0], [-0.2, 0.1, 1.0]])
    k = k / np.linalg.norm(k, axis=1, keepdims=True)
    kw = dict(interpolation=1, case_type=1, kvectors=k)
    for phys in (5.0, 1.2):
        ref = O.simulate(O.Sim(dims, 2, phys, energies, angles, **kw), vox, mats)
        sim = capi.Sim(dims, 2, phys, energies, angles, precision=capi.FP64, pipeline=capi.PIPE_EBASIS, **kw)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < 1e-10, (phys, err)
