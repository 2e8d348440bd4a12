"""The any-length X kernel with its outputs split over blocks or run one after another, on
both sides of the line (98304 threads of rows), in every mode and precision.  Bars as in every
parity test."""
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

pytest.importorskip("torch")


# threads: rows x ceil(Nx / 4) in FP32, / 2 in FP64
@pytest.mark.gpu
@pytest.mark.parametrize("prec,dims", [(capi.FP64, (90, 70, 12)), (capi.FP64, (90, 70, 31)), (capi.FP64, (90, 70, 32)),
                                       (capi.FP32, (90, 70, 60)), (capi.FP32, (90, 70, 61))])
def test_x_outputs_split_or_not(prec, dims):
    print(f"x split {dims} prec={prec}", flush=True)
    energies, angles = [285.0], (0.0, 60.0, 120.0)
    for M in (1, 2):  # single, pair; the E-basis: tensor
        vox, mats = random_euler(dims, M, 61), random_constants(1, M, 62)
        kw = dict(interpolation=1, windowing=1)
        ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
        for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
            sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=pipeline, **kw)
            err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
            assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), (M, pipeline, err)
