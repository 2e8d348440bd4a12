"""The plain executor's E-angle batches where their buffers do not fit: one angle at a time."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from tests.helpers import random_constants, random_euler

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [{}, dict(algorithm=1), dict(scatter_approach=1)])
def test_batches_give_way(kw, monkeypatch):
    dims, M, V = (30, 32, 12), 2, 30 * 32 * 12
    print(f"plain memory {kw}", flush=True)
    vox, mats = random_euler(dims, M, 4), random_constants(2, M, 5)
    sim = capi.Sim(dims, M, 3.0, [283.0, 286.0], (0.0, 20.0, 160.0), pipeline=capi.PIPE_PLAIN, interpolation=1, **kw)
    ref = capi.simulate(sim, vox, mats)
    capi.lib().cyr_release_workspace()
    # room for the morphology, one angle's three volumes and Algorithm 1's six, not for eight
    # angles' 24
    monkeypatch.setenv("CYR_TEST_FAIL_ALLOC", f">{8 * V * 6}")
    got = capi.simulate(sim, vox, mats)
    err = np.nanmax(np.abs(got - ref)) / np.nanmax(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and err < 1e-6, err
