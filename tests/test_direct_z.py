"""Stacks whose Z pencil fits in LDS but no convolution for it does (more than 8192 points,
FP64 5120, with a large prime factor): fused executors, the Z pass by the direct sum."""
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

torch = pytest.importorskip("torch")

# (64 rows in FP32: the E-basis by the fused Y / z-bin kernel, 3: by separate passes)
CASES = [(capi.FP32, (4, 3, 8209), 0), (capi.FP32, (4, 3, 8209), 1), (capi.FP32, (2, 64, 8209), 1),
         (capi.FP64, (4, 3, 5147), 0), (capi.FP64, (4, 3, 5147), 1)]


@pytest.mark.parametrize("prec,dims", [c[:2] for c in CASES[1::2] + CASES[2:3]] +
                         [(capi.FP32, (64, 64, 20479)), (capi.FP64, (32, 32, 10223))])
def test_long_stacks_are_fused(prec, dims):
    for pipeline in (capi.PIPE_EBASIS, capi.PIPE_MBASIS):
        sim = capi.Sim(dims, 2, 2.0, [285.0, 286.0], (0, 30, 150), precision=prec, pipeline=pipeline)
        assert sim.resolved_pipeline() == pipeline


@pytest.mark.gpu
@pytest.mark.parametrize("prec,dims,interpolation", CASES)
def test_long_stacks_match_the_oracle(prec, dims, interpolation):
    """Bars as in every parity test (FP64 1e-10, FP32 1e-4, identical masks)."""
    print(f"direct Z {dims} prec={prec} interpolation={interpolation}", flush=True)
    M, energies, angles = 2, [283.0, 287.0][:1 + (dims[1] < 64)], (0.0, 60.0, 60.0 * (dims[1] < 64))
    vox, mats = random_euler(dims, M, 51), random_constants(len(energies), M, 52)
    kw = dict(interpolation=interpolation, windowing=1)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=pipeline, **kw)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), (dims, pipeline, err)
