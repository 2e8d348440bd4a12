"""Captured plans: members whose own executors do not fit the device (the plan runs the
executor that the eager call falls back to), and members of more units than the process
keeps band widths for."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from tests.helpers import random_constants, random_euler

torch = pytest.importorskip("torch")

# (grid, materials, energies, executor asked for, executor that fits, its larger buffers'
# bytes): limits between the two executors' largest buffer
CASES = {
    # 7 packed volumes of 8 bytes a voxel against plain's 3
    "mbasis_to_plain": ((50, 50, 40), 4, 2, capi.PIPE_MBASIS, capi.PIPE_PLAIN, 5 * 8 * 50 * 50 * 40),
    # two rows or more of 28 band values of 8 bytes a pixel against the E-basis' partial sums
    # of at most 5 chunks x 2 bins x 5 fields
    "auto_to_ebasis": ((256, 512, 5), 4, 20, capi.PIPE_AUTO, capi.PIPE_EBASIS, 53 * 8 * 256 * 512),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_plan_falls_back_as_the_eager_call(case, monkeypatch):
    dims, M, nE, asked, fits, limit = CASES[case]
    print(f"plan fallback {case}", flush=True)
    V, energies = dims[0] * dims[1] * dims[2], [285.0 + i for i in range(nE)]
    vox = torch.from_numpy(random_euler(dims, M, 5).astype(np.float32)).cuda()
    small_vox = torch.from_numpy(random_euler((32, 32, 16), 2, 6).astype(np.float32)).cuda()
    mats, small_mats = random_constants(nE, M, 7), random_constants(2, 2, 8)
    mk = lambda pipe: capi.Sim(dims, M, 2.0, energies, (0, 5, 175), pipeline=pipe, interpolation=1)
    small = capi.Sim((32, 32, 16), 2, 2.0, [284.0, 286.0], (0, 30, 150), pipeline=capi.PIPE_AUTO, interpolation=1)
    out = lambda n, d: torch.empty((n, 1, d[1], d[0]), device="cuda")
    ref, small_ref = out(nE, dims), out(2, (32, 32))
    capi.simulate_device(mk(fits), vox, mats, ref)
    capi.simulate_device(small, small_vox, small_mats, small_ref)
    assert mk(asked).resolved_pipeline() == capi.PIPE_MBASIS
    outs = [out(2, (32, 32)), out(nE, dims), out(nE, dims)]
    monkeypatch.setenv("CYR_TEST_FAIL_ALLOC", f">{limit}")
    # one stream: its members share the buffers that a fallback frees
    plan = capi.BatchPlan([small, mk(asked), mk(asked)], [small_vox, vox, vox], [small_mats, mats, mats], outs, lanes=1)
    try:
        for rep in range(3):
            for o in outs:
                o.fill_(0.0)
            plan.launch()
            torch.cuda.synchronize()
            for o, r in zip(outs, (small_ref, ref, ref)):
                np.testing.assert_array_equal(o.cpu().numpy(), r.cpu().numpy())
    finally:
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("pipeline,prec,nE,nK", [(capi.PIPE_EBASIS, capi.FP64, 4200, 1), (capi.PIPE_MBASIS, capi.FP32, 1, 4200)])
def test_plan_of_many_units(pipeline, prec, nE, nK):
    """More than 4096 (energy, k vector) units in one plan: its replays equal the eager call."""
    print(f"plan of many units pipeline={pipeline}", flush=True)
    dims, M = (10, 8, 6), 2
    dt = torch.float64 if prec == capi.FP64 else torch.float32
    energies = list(np.linspace(280.0, 300.0, nE))
    tilt = np.linspace(0.0, 0.05, nK)
    kv = np.stack([np.sin(tilt), np.zeros(nK), np.cos(tilt)], axis=1) if nK > 1 else None
    vox = torch.from_numpy(random_euler(dims, M, 15)).to(dt).cuda()
    mats = random_constants(nE, M, 16)
    sim = capi.Sim(dims, M, 3.0, energies, (0, 90, 90), precision=prec, pipeline=pipeline, interpolation=1,
                   **({"kvectors": kv, "case_type": 1} if nK > 1 else {}))
    assert sim.resolved_pipeline() == pipeline
    ref, out = (torch.empty((nE, nK, dims[1], dims[0]), dtype=dt, device="cuda") for _ in range(2))
    capi.simulate_device(sim, vox, mats, ref)
    plan = capi.BatchPlan([sim], [vox], [mats], [out], lanes=1)
    try:
        for rep in range(2):
            out.fill_(0.0)
            plan.launch()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(out.cpu().numpy(), ref.cpu().numpy())
    finally:
        plan.close()
