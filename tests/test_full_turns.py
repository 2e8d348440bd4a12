"""Whole-turn angle lists: the rotation sums each angle's quarter turns before it samples.
Against the oracle, at the edges of its rule: fewer angles per quarter than waves, more
than one run of 64, planes whose quarter is no multiple of a tile or of 4, the Ewald disc
inside the plane and past its corners, the mask, tilted beams (whose discs are not their
own quarter turn), base angles off the pixel axes, and angles on multiples of 90 and 45
degrees (points on pixel edges).  Bars: FP64 1e-10, FP32 1e-4, identical masks."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")

TILT = np.array([[0.0, 0.25, 1.0], [-0.2, 0.1, 1.0]])
TILT = TILT / np.linalg.norm(TILT, axis=1, keepdims=True)

CASES = {
    # (dims, energies, angles, phys, options)
    "four_angles": ((128, 128, 1), 34, (0.0, 90.0, 270.0), 2.0, {}),
    "disc_inside": ((128, 128, 1), 34, (0.0, 15.0, 345.0), 1.0, {}),
    "disc_inside_mask": ((130, 130, 1), 34, (0.0, 15.0, 345.0), 1.0, dict(rot_mask=1)),
    "past_corners_mask": ((134, 134, 1), 33, (7.5, 22.5, 345.0), 5.0, dict(rot_mask=1)),
    "past_corners": ((156, 156, 1), 22, (3.0, 9.0, 354.0), 5.0, {}),
    "three_d": ((96, 96, 4), 60, (0.0, 10.0, 350.0), 2.0, dict(windowing=1)),
    "long_runs": ((128, 128, 1), 33, (0.0, 0.25, 359.75), 1.5, dict(rot_mask=1)),
    "tilted": ((128, 128, 1), 33, (0.0, 30.0, 330.0), 1.0, dict(case_type=1, kvectors=TILT)),
    "tilted_mask": ((128, 128, 1), 33, (0.0, 30.0, 330.0), 1.0, dict(case_type=1, kvectors=TILT, rot_mask=1)),
}


@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("case", sorted(CASES))
def test_full_turns(case, prec):
    dims, nE, angles, phys, kw = CASES[case]
    print(f"full turns {case} prec={prec}", flush=True)
    vox = random_euler(dims, 2, 21)
    energies = list(280.0 + 0.25 * np.arange(nE))
    mats = random_constants(nE, 2, 22)
    kw = dict(kw, interpolation=1)
    ref = O.simulate(O.Sim(dims, 2, phys, energies, angles, **kw), vox, mats)
    sim = capi.Sim(dims, 2, phys, energies, angles, precision=prec, pipeline=capi.PIPE_MBASIS, **kw)
    err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
    print(f"  rel L2 {err:.3e}")
    assert same, case
    assert err < (1e-10 if prec == capi.FP64 else 1e-4), (case, err)


def test_full_turns_nan():
    """NaN in the morphology reaches every value: the same pixels are finite as with the
    per-angle executor."""
    dims, nE, angles = (128, 128, 1), 33, (0.0, 30.0, 330.0)
    energies = list(280.0 + 0.25 * np.arange(nE))
    mats = random_constants(nE, 2, 22)
    vox = random_euler(dims, 2, 21).astype(np.float32)
    vox.reshape(2, -1, 4)[0, 40, 0] = np.nan
    for rot_mask in (0, 1):
        got = []
        for pipeline in (capi.PIPE_MBASIS, capi.PIPE_PLAIN):
            sim = capi.Sim(dims, 2, 1.0, energies, angles, pipeline=pipeline, interpolation=1, rot_mask=rot_mask)
            got.append(np.isfinite(capi.simulate(sim, vox, mats)))
        np.testing.assert_array_equal(got[0], got[1])
