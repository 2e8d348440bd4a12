"""Which E-basis passes FP64 grids run, and which executor AUTO gives way to where its
own buffers exceed a limit."""
import ctypes

import numpy as np
import pytest

from cyrsoxs_amd import capi
from tests.helpers import pattern_rel_l2, random_constants

torch = pytest.importorskip("torch")


def _gate(sim):
    """Status of the allocation-free call's size gate (7, no device: the request passed)."""
    buf = np.zeros(64)
    p = ctypes.c_void_p(buf.ctypes.data)
    return capi.lib().cyr_simulate_device_noalloc(sim.ref, p, p, p, None)


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the gate alone, on host pointers")
def test_auto_gives_way_to_the_e_basis():
    energies = [285.0 + i for i in range(20)]
    mk = lambda pipe, dims=(256, 512, 5): capi.Sim(dims, 4, 2.0, energies, (0, 5, 175), pipeline=pipe, interpolation=1)
    assert mk(capi.PIPE_AUTO).resolved_pipeline() == capi.PIPE_MBASIS
    assert _gate(mk(capi.PIPE_MBASIS)) == 1
    assert _gate(mk(capi.PIPE_AUTO)) == 7
    # where the volumes dominate, the material basis is what the bytes prefer too
    assert _gate(mk(capi.PIPE_AUTO, (128, 128, 128))) == 1


@pytest.mark.gpu
def test_auto_in_scratch_is_the_e_basis():
    dims, M, energies = (256, 512, 5), 4, [285.0 + i for i in range(20)]
    vox = torch.rand((M, 256 * 512 * 5, 4), generator=torch.Generator().manual_seed(2)).cuda()
    mats, out = random_constants(20, M, 4), {}
    for pipe in (capi.PIPE_AUTO, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 2.0, energies, (0, 5, 175), pipeline=pipe, interpolation=1)
        out[pipe] = torch.empty((20, 1, 512, 256), device="cuda")
        capi.simulate_device_noalloc(sim, vox, mats, out[pipe])
    np.testing.assert_array_equal(out[capi.PIPE_AUTO].cpu().numpy(), out[capi.PIPE_EBASIS].cpu().numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(256, 256, 103), (256, 256, 102), (16, 512, 9), (30, 64, 2)])
def test_fp64_e_basis_either_pass(dims):
    """Both sides of the line between the fused Y/z kernel and the separate passes: the
    material basis within twice the FP64 bar of 1e-10 against the oracle."""
    M, energies = 2, [284.0, 287.0]
    n = dims[0] * dims[1] * dims[2]
    print(f"fp64 E-basis {dims}", flush=True)
    vox = torch.rand((M, n, 4), generator=torch.Generator().manual_seed(9), dtype=torch.float64).cuda()
    mats, got = random_constants(2, M, 4), {}
    for pipe in (capi.PIPE_MBASIS, capi.PIPE_EBASIS):
        sim = capi.Sim(dims, M, 2.0, energies, (0, 60, 120), precision=capi.FP64, pipeline=pipe, interpolation=1)
        out = torch.empty((2, 1, dims[1], dims[0]), dtype=torch.float64, device="cuda")
        capi.simulate_device(sim, vox, mats, out)
        torch.cuda.synchronize()
        got[pipe] = out.cpu().numpy()
    err, same = pattern_rel_l2(got[capi.PIPE_EBASIS], got[capi.PIPE_MBASIS])
    assert same and err < 2e-10, err
