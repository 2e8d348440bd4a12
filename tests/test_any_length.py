"""Sides without a compile-time codelet: the any-length transforms (lfft.hpp) as
single passes and inside the fused executors, which take them on every grid.

Lengths cover each radix alone (2 ... 13), products of several, primes that run
Bluestein's algorithm from the shortest (17) up, tiles of fewer columns, and pencils
longer than a thread block's first round.  FP32 transforms: a pencil of up to 4096
convolution points loses at most about 12 x 0.6 x 6e-8 per transform, two of them and
three products per axis, three axes: 4e-6.  Patterns keep the bars of every other
parity test (FP64 1e-10, FP32 1e-4 of the FP64 oracle, identical NaN masks).
"""
import ctypes

import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler, random_vector, rel_l2

torch = pytest.importorskip("torch")

# (nx, ny, nz): every axis meets the lengths in turn
FFT_SHAPES = [(2, 3, 5), (4, 6, 7), (8, 9, 10), (11, 13, 2), (17, 19, 23), (29, 31, 37), (101, 4, 47), (5, 94, 21),
              (200, 12, 50), (12, 240, 3), (3, 250, 96), (121, 6, 143), (169, 5, 1), (2, 499, 3), (499, 2, 2),
              (3, 2, 997), (1000, 3, 2), (4, 1000, 1), (1500, 2, 1), (2, 1021, 1), (1021, 2, 1), (2, 1620, 1),
              (2, 3000, 1), (3, 2, 2187)]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("dims", FFT_SHAPES)
def test_fft3d_any_length(dims, prec):
    nx, ny, nz = dims
    print(f"any-length fft3d dims={dims} prec={prec}", flush=True)
    rng = np.random.default_rng(nx * 7 + ny * 3 + nz)
    vols = [rng.normal(size=(nz, ny, nx)) + 1j * rng.normal(size=(nz, ny, nx)) for _ in range(2)]
    dev = [torch.from_numpy(v.astype(np.complex128 if prec == capi.FP64 else np.complex64)).cuda() for v in vols]
    capi.fft3d_device(dev, dims, prec)
    torch.cuda.synchronize()
    for v, d in zip(vols, dev):
        err = rel_l2(d.cpu().numpy(), np.fft.fftn(v))
        assert err < (1e-12 if prec == capi.FP64 else 4e-6), (dims, prec, err)


CASES = {
    # (dims, M, morphology, options, PhysSize)
    "prime_sides": ((17, 19, 23), 2, 0, dict(interpolation=1, windowing=1), 5.0),
    "cut_sides": ((53, 46, 21), 3, 0, dict(interpolation=1), 2.0),
    "round_sides": ((50, 60, 20), 2, 1, dict(interpolation=0, windowing=1), 2.0),
    "radices_11_13": ((22, 26, 33), 1, 0, dict(interpolation=1), 1.4),
    "film_prime": ((61, 59, 1), 3, 0, dict(interpolation=1), 1.0),
    "film_round_mask": ((100, 90, 1), 2, 1, dict(interpolation=0, rot_mask=1), 1.0),
    "material_frame": ((40, 35, 14), 2, 0, dict(interpolation=1, reference_frame=0, rot_mask=1), 1.6),
    "wide_rows": ((230, 20, 6), 2, 0, dict(interpolation=1, windowing=1), 5.0),
    "long_columns": ((12, 310, 5), 2, 1, dict(interpolation=1), 2.0),
    "short_z": ((32, 48, 2), 2, 0, dict(interpolation=0), 5.0),
    "mixed_codelets": ((64, 50, 128), 2, 0, dict(interpolation=1, windowing=1), 1.5),
}


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("case", sorted(CASES))
def test_fused_executors_any_grid(case, prec):
    dims, M, morph, kw, phys = CASES[case]
    print(f"any grid {case} {dims} prec={prec}", flush=True)
    vox = random_euler(dims, M, 5) if morph == 0 else random_vector(dims, M, 5)
    energies = [282.0, 285.5, 289.0]
    mats = random_constants(len(energies), M, 6)
    kw = dict(kw, morphology_type=morph)
    angles = (0.0, 15.0, 165.0)
    ref = O.simulate(O.Sim(dims, M, phys, energies, angles, **kw), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS, capi.PIPE_PLAIN):
        sim = capi.Sim(dims, M, phys, energies, angles, precision=prec, pipeline=pipeline, **kw)
        assert sim.resolved_pipeline() == pipeline
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        print(f"  pipeline {pipeline}: rel L2 {err:.3e}")
        assert same, (case, pipeline)
        assert err < (1e-10 if prec == capi.FP64 else 1e-4), (case, pipeline, err)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [capi.STORE_FP16, capi.STORE_BF16])
def test_any_grid_16_bit_storage(storage):
    """The any-length X kernel's 16-bit morphology loads: the same bars as on the grids
    with codelets (10x the storage error measured there)."""
    dims, M = (50, 34, 18), 3
    vox, energies = random_euler(dims, M, 31), [284.0, 286.0]
    mats = random_constants(2, M, 5)
    kw = dict(interpolation=1, windowing=1)
    ref = O.simulate(O.Sim(dims, M, 5.0, energies, (0, 30, 150), **kw), vox, mats)
    for pipeline in (capi.PIPE_EBASIS, capi.PIPE_MBASIS):
        sim = capi.Sim(dims, M, 5.0, energies, (0, 30, 150), storage=storage, pipeline=pipeline, **kw)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < (1e-4 if storage == capi.STORE_FP16 else 4e-4), err


def _noalloc(sim):
    """Status of the size gate (no device here: a request that passes it reports that)."""
    buf = np.zeros(64)
    p = ctypes.c_void_p(buf.ctypes.data)
    return capi.lib().cyr_simulate_device_noalloc(sim.ref, p, p, p, None)


def test_routes_of_other_grids():
    """Every grid of ordinary sides resolves to a fused executor; sides below 8 with a
    larger prime factor stay plain."""
    for dims in ((100, 100, 100), (101, 94, 21), (31, 17, 1), (1000, 500, 1), (2039, 2039, 1), (7 * 13, 97, 8)):
        for prec in (capi.FP32, capi.FP64):
            sim = capi.Sim(dims, 3, 2.0, list(np.linspace(280, 299, 20)), (0, 5, 175), precision=prec,
                           pipeline=capi.PIPE_AUTO)
            assert sim.resolved_pipeline() in (capi.PIPE_EBASIS, capi.PIPE_MBASIS), (dims, prec)
    for dims in ((7, 16, 16), (16, 7, 16), (16, 16, 7)):
        assert capi.Sim(dims, 1, 2.0, [280.0], (0, 5, 175),
                        pipeline=capi.PIPE_MBASIS).resolved_pipeline() == capi.PIPE_PLAIN


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the gate alone, on host pointers")
def test_scratch_limit_keeps_its_callers():
    """A grid that had only the plain executor keeps running in the scratch array when the
    fused executor's buffers exceed it; one that always had a fused executor is still
    rejected."""
    energies = list(np.linspace(280, 299, 20))
    was_plain = capi.Sim((130, 130, 110), 4, 2.0, energies, (0, 5, 175), pipeline=capi.PIPE_MBASIS)
    assert was_plain.resolved_pipeline() == capi.PIPE_MBASIS
    assert _noalloc(was_plain) == 7  # past the gate: no device
    was_fused = capi.Sim((128, 128, 128), 4, 2.0, energies, (0, 5, 175), pipeline=capi.PIPE_MBASIS)
    assert _noalloc(was_fused) == 1


@pytest.mark.gpu
def test_scratch_limit_falls_back_to_plain():
    """The same on the device: the patterns of the plain executor."""
    dims, M, energies, angles = (130, 130, 110), 2, [282.0, 285.0], (0.0, 45.0, 90.0)
    rng = torch.Generator().manual_seed(3)
    vox = torch.rand((M, dims[0] * dims[1] * dims[2], 4), generator=rng).cuda()
    mats = random_constants(len(energies), M, 8)
    kw = dict(interpolation=1, windowing=1)
    out = {}
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_PLAIN):
        sim = capi.Sim(dims, M, 2.0, energies, angles, pipeline=pipeline, **kw)
        out[pipeline] = torch.empty((2, 1, dims[1], dims[0]), dtype=torch.float32, device="cuda")
        capi.simulate_device_noalloc(sim, vox, mats, out[pipeline])
    a, b = (out[p].cpu().numpy() for p in (capi.PIPE_MBASIS, capi.PIPE_PLAIN))
    assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.gpu
def test_engine_budget_falls_back_to_plain():
    """A request whose fused footprint exceeds the engine's budget but whose plain one
    fits is admitted, as it was when its grid had no fused executor."""
    dims, M, energies, angles = (50, 50, 50), 4, [282.0, 285.0], (0.0, 45.0, 90.0)
    vox = random_euler(dims, M, 9)
    mats = random_constants(len(energies), M, 8)
    kw = dict(interpolation=1, windowing=1)
    fused = capi.Sim(dims, M, 2.0, energies, angles, pipeline=capi.PIPE_MBASIS, **kw)
    plain = capi.Sim(dims, M, 2.0, energies, angles, pipeline=capi.PIPE_PLAIN, **kw)
    assert plain.footprint() < fused.footprint()
    ref = capi.simulate(plain, vox, mats)
    with capi.Engine(budget_bytes=plain.footprint() + 1024, slots=1) as eng:
        rid = eng.submit(fused, vox, mats)
        assert eng.wait(rid) == 0
        assert np.array_equal(eng.result(rid), ref, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("dims", [(143, 10, 4), (9, 9, 1), (10, 50, 3), (1100, 4, 1), (1030, 6, 2), (2310, 4, 1),
                                  (2048, 6, 1)])
def test_x_rows_of_every_plan(dims, prec):
    """Rows of the X kernel by each of its plans: radices up to 8, factors 11 and 13 (a
    wide plan in FP32, Bluestein in FP64), the longer per-thread runs of long rows; several
    rows a block with the last block short.  Bars as above."""
    if prec == capi.FP64 and dims[0] > 2048:
        pytest.skip("longer than the FP64 row limit")
    print(f"X rows {dims} prec={prec}", flush=True)
    M, energies, angles = 2, [283.0, 287.0], (0.0, 60.0, 120.0)
    vox, mats = random_euler(dims, M, 12), random_constants(2, M, 13)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, interpolation=1, windowing=1), vox, mats)
    for pipeline in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=pipeline, interpolation=1, windowing=1)
        err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
        assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), (dims, pipeline, err)
