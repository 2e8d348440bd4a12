"""Columns so long that the any-length Y pass has one or two of them in a tile: the sums of
the DC replacement's neighbours come from columns 0, 1 and Nx - 1, which then lie in three
blocks.  Every simulation here follows one that leaves values 1e6 times larger in the work
buffers.  Bars as in every parity test (FP64 1e-10, FP32 1e-4 of the FP64 oracle, identical
masks), for the pattern and for the nine pixels about its centre, which the replaced value
dominates.
"""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler, random_vector

torch = pytest.importorskip("torch")

# one column a tile: Bluestein sides from 1621 (FP64) and 3001 (FP32) on, 3200 = 2^7 5^2 in
# FP64; two: 1500 in FP64, 2310 in FP32
CASES = [(capi.FP64, (12, 1621, 1)), (capi.FP64, (10, 1999, 2)), (capi.FP64, (6, 3200, 2)), (capi.FP64, (3, 1700, 1)),
         (capi.FP64, (8, 1500, 2)), (capi.FP32, (8, 3001, 1)), (capi.FP32, (6, 3010, 2)), (capi.FP32, (9, 2310, 2))]


def _dirty(prec):
    vox = random_vector((64, 64, 32), 4, 3) * 1e3
    sim = capi.Sim((64, 64, 32), 4, 2.0, [285.0], (0, 30, 60), precision=prec, morphology_type=1,
                   pipeline=capi.PIPE_MBASIS)
    capi.simulate(sim, vox, random_constants(1, 4, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("prec,dims", CASES)
def test_dc_sums_of_narrow_tiles(prec, dims):
    print(f"narrow tiles {dims} prec={prec}", flush=True)
    M, energies, angles = 2, [283.0, 287.0], (0.0, 60.0, 120.0)
    vox, mats = random_euler(dims, M, 21), random_constants(2, M, 22)
    kw = dict(interpolation=1, rot_mask=1)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
    bar = 1e-10 if prec == capi.FP64 else 1e-4
    cx, cy = dims[0] // 2, dims[1] // 2
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=pipeline, **kw)
        assert sim.resolved_pipeline() == pipeline
        _dirty(prec)
        got = capi.simulate(sim, vox, mats)
        err, same = pattern_rel_l2(got, ref)
        assert same and err < bar, (dims, pipeline, err)
        box = (..., slice(cy - 1, cy + 2), slice(max(0, cx - 1), cx + 2))
        err, same = pattern_rel_l2(got[box], ref[box])
        assert same and err < bar, (dims, pipeline, "centre", err)
