"""Grids that run the fused executors: stacks of seven planes."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

torch = pytest.importorskip("torch")


def _resolved(dims, prec, pipeline):
    return capi.Sim(dims, 2, 2.0, list(np.linspace(280, 299, 20)), (0, 5, 175), precision=prec,
                    pipeline=pipeline).resolved_pipeline()


@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("dims", [(128, 128, 7), (512, 512, 7), (2048, 1024, 7), (17, 16, 7), (250, 90, 7)])
def test_seven_planes_are_fused(dims, prec):
    for pipeline in (capi.PIPE_EBASIS, capi.PIPE_MBASIS):
        assert _resolved(dims, prec, pipeline) == pipeline
    assert _resolved(dims, prec, capi.PIPE_AUTO) != capi.PIPE_PLAIN


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("dims", [(40, 36, 7), (64, 64, 7)])
def test_seven_planes_match_the_oracle(dims, prec):
    """Bars as in every parity test."""
    print(f"seven planes {dims} prec={prec}", flush=True)
    M, energies, angles = 3, [283.0, 287.0], (0.0, 30.0, 150.0)
    vox, mats = random_euler(dims, M, 41), random_constants(2, M, 42)
    kw = dict(interpolation=1, windowing=1)
    ref = O.simulate(O.Sim(dims, M, 2.0, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS, capi.PIPE_AUTO):
        sim = capi.Sim(dims, M, 2.0, energies, angles, precision=prec, pipeline=pipeline, **kw)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), (dims, pipeline, err)
