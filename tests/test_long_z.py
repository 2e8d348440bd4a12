"""Long columns: tiles of the Z band pass that fill the 160 KB of LDS, and Y and Z columns
whose tables stay in memory.  Bars as in every parity test (FP64 1e-10, FP32 1e-4 of the
FP64 oracle, identical masks)."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler, rel_l2

torch = pytest.importorskip("torch")

# FP64 2048: the codelet's four columns take the LDS whole; 1944, 3125 and FP32 4460, 8100:
# any-length tiles within 256 bytes of it
CASES = [(capi.FP64, (12, 8, 2048)), (capi.FP64, (8, 10, 1944)), (capi.FP64, (6, 4, 3125)), (capi.FP32, (8, 6, 4460)),
         (capi.FP32, (6, 4, 8100)),
         # tables in memory
         (capi.FP64, (6, 4, 5000)), (capi.FP32, (4, 4, 9216)), (capi.FP32, (3, 9216, 1)), (capi.FP32, (4, 8192, 2)),
         (capi.FP64, (3, 8192, 1))]


@pytest.mark.gpu
@pytest.mark.parametrize("prec,dims", CASES)
def test_long_columns(prec, dims):
    print(f"long columns {dims} prec={prec}", flush=True)
    M, energies, angles = 2, [283.0, 287.0], (0.0, 60.0, 120.0)
    vox, mats = random_euler(dims, M, 31), random_constants(2, M, 32)
    kw = dict(interpolation=1, windowing=1)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=pipeline, **kw)
        assert sim.resolved_pipeline() == pipeline
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), (dims, pipeline, err)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(2, 18432, 1), (18432, 2, 1), (3, 20480, 1), (20480, 2, 1), (2, 2, 16875)])
def test_transforms_longer_than_16384(dims):
    """One FP32 pencil of up to 20480 points in LDS (tolerance as for the shorter lengths: 15
    roundings of 6e-8 a butterfly, five stages, two axes, below 4e-6)."""
    print(f"fft3d {dims}", flush=True)
    rng = np.random.default_rng(dims[0] + dims[1])
    v = rng.normal(size=dims[::-1]) + 1j * rng.normal(size=dims[::-1])
    d = torch.from_numpy(v.astype(np.complex64)).cuda()
    capi.fft3d_device([d], dims, capi.FP32)
    torch.cuda.synchronize()
    assert rel_l2(d.cpu().numpy(), np.fft.fftn(v)) < 4e-6


@pytest.mark.parametrize("prec,dims", [(capi.FP32, (64, 64, 16000)), (capi.FP32, (64, 8192, 64)),
                                       (capi.FP32, (64, 12288, 1)), (capi.FP64, (64, 64, 10000)),
                                       (capi.FP64, (64, 8192, 1))])
def test_long_columns_are_fused(prec, dims):
    sim = capi.Sim(dims, 2, 2.0, [285.0, 286.0], (0, 30, 150), precision=prec, pipeline=capi.PIPE_MBASIS)
    assert sim.resolved_pipeline() == capi.PIPE_MBASIS
