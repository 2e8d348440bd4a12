"""E-basis, laboratory frame, FP32: an angle's intensity where the quadratic form's terms
cancel.

One material aligned along (1, 1, 0) with n_perp = 1: N = d w s s^T, so the intensity of E at
angle theta goes with (cos theta + sin theta)^2.  The eleven angles 134.8 ... 135.2 degrees
average to 8e-6 of the form's components: components rounded to FP32 (6e-8) leave about
7e-3 of the average, projections of each angle about 3e-5, FP64 forms of the same fields
less.  Bar as in every FP32 parity test, 1e-4 of the FP64 oracle.
"""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2

pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(64, 64, 16), (48, 50, 12), (64, 64, 1), (40, 36, 1)])
def test_cancelling_forms(dims):
    print(f"cancelling forms {dims}", flush=True)
    V = dims[0] * dims[1] * dims[2]
    w = np.random.default_rng(3).uniform(0.2, 1.0, V).astype(np.float32)
    vox = np.zeros((1, V, 4))
    vox[0, :, 0] = vox[0, :, 1] = w
    mats = np.array([[[1 - 1e-3, 1e-3, 1.0, 0.0]], [[1 - 2e-3, 5e-4, 1.0, 0.0]]])
    args = (dims, 1, 2.0, [284.0, 287.0], (134.8, 0.04, 135.2))
    kw = dict(interpolation=1, windowing=1, morphology_type=1)
    ref = O.simulate(O.Sim(*args, **kw), vox, mats)
    sim = capi.Sim(*args, pipeline=capi.PIPE_EBASIS, **kw)
    assert sim.num_angles == 11 and sim.resolved_pipeline() == capi.PIPE_EBASIS
    err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
    assert same and err < 1e-4, (dims, err)
