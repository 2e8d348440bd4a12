"""Grids that run the fused executors: stacks of seven planes, FP32 rows of 4097 to 8192
points."""
import ctypes

import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler, random_vector

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


@pytest.mark.parametrize("nx", [4608, 5184, 5832, 6144])
def test_long_rows_are_fused(nx):
    for dims in ((nx, 64, 1), (nx, 96, 12)):
        for pipeline in (capi.PIPE_EBASIS, capi.PIPE_MBASIS):
            assert _resolved(dims, capi.FP32, pipeline) == pipeline


@pytest.mark.gpu
@pytest.mark.parametrize("nx,M,morph", [(4100, 2, 0), (4608, 1, 0), (6144, 2, 0), (6144, 3, 1), (8192, 2, 0)])
def test_long_rows_match_the_oracle(nx, M, morph):
    """The X kernel's longest runs per thread (FP32, 1e-4 of the oracle, identical masks)."""
    dims, energies, angles = (nx, 4, 2), [283.0, 287.0], (0.0, 60.0, 120.0)
    print(f"long rows {dims} M={M} morph={morph}", flush=True)
    vox, mats = (random_vector if morph else random_euler)(dims, M, 43), random_constants(2, M, 44)
    kw = dict(interpolation=1, windowing=1, rot_mask=1, morphology_type=morph)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 3.0, energies, angles, precision=capi.FP32, pipeline=pipeline, **kw)
        assert sim.resolved_pipeline() == pipeline
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < 1e-4, (dims, pipeline, err)


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the gate alone, on host pointers")
@pytest.mark.parametrize("dims,prec,status", [
    # rows of 3^7, 5^5 and 2 3^7 points, and columns of 4 3^7, need more threads than the short
    # radix plans have: past the gate with the plain executor's buffers (7: no device)
    ((2187, 64, 24), capi.FP32, 7), ((3125, 64, 16), capi.FP32, 7), ((4374, 32, 24), capi.FP32, 7),
    ((48, 8748, 8), capi.FP32, 7), ((16, 6561, 24), capi.FP32, 7), ((130, 130, 200), capi.FP32, 7),
    # sides with short plans: refused (1)
    ((2048, 64, 24), capi.FP32, 1), ((3072, 64, 16), capi.FP32, 1), ((48, 4096, 20), capi.FP32, 1),
    ((81, 243, 150), capi.FP32, 1), ((125, 625, 40), capi.FP32, 1), ((144, 128, 160), capi.FP32, 1)])
def test_requests_that_do_not_fit(dims, prec, status):
    sim = capi.Sim(dims, 4, 2.0, [285.0, 286.0], (0, 5, 175), precision=prec, pipeline=capi.PIPE_MBASIS)
    assert sim.resolved_pipeline() == capi.PIPE_MBASIS
    buf = np.zeros(64)
    p = ctypes.c_void_p(buf.ctypes.data)
    assert capi.lib().cyr_simulate_device_noalloc(sim.ref, p, p, p, None) == status
