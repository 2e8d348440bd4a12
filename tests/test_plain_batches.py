"""The plain executor's batches of E angles (small grids take up to 8 per launch): angle
counts on both sides of a batch, Algorithm 1, the material frame, the rotation mask, and
the full projection, which stays at one angle.  A batched run and the one-angle run of
the same simulation (through cyr_simulate_batch, which keeps single angles) agree to
rounding; both meet the oracle's bars."""
import numpy as np
import pytest

from cyrsoxs_amd import capi
from oracle import oracle as O
from tests.helpers import pattern_rel_l2, random_constants, random_euler

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = {
    "one": ((0.0, 1.0, 0.0), {}),
    "seven": ((0.0, 20.0, 120.0), dict(rot_mask=1)),
    "eight": ((0.0, 20.0, 140.0), dict(reference_frame=0)),
    "nine_alg1": ((0.0, 20.0, 160.0), dict(algorithm=1)),
    "alg1_material": ((0.0, 10.0, 170.0), dict(algorithm=1, reference_frame=0)),
    "full": ((0.0, 20.0, 160.0), dict(scatter_approach=1)),
}


@pytest.mark.parametrize("prec", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("case", sorted(CASES))
def test_plain_angle_batches(case, prec):
    angles, kw = CASES[case]
    dims, M, energies = (32, 30, 12), 2, [283.0, 286.0]
    print(f"plain batches {case} prec={prec}", flush=True)
    vox, mats = random_euler(dims, M, 4), random_constants(2, M, 5)
    kw = dict(kw, interpolation=1, windowing=1)
    ref = O.simulate(O.Sim(dims, M, 3.0, energies, angles, **kw), vox, mats)
    sim = capi.Sim(dims, M, 3.0, energies, angles, precision=prec, pipeline=capi.PIPE_PLAIN, **kw)
    got = capi.simulate(sim, vox, mats)
    dt = torch.float64 if prec == capi.FP64 else torch.float32
    out = torch.empty((2, 1, dims[1], dims[0]), dtype=dt, device="cuda")
    capi.simulate_batch([sim], [torch.from_numpy(vox).to(dt).cuda()], [mats], [out])
    for g in (got, out.cpu().numpy()):
        err, same = pattern_rel_l2(g, ref)
        assert same and err < (1e-10 if prec == capi.FP64 else 1e-4), err
    err, same = pattern_rel_l2(got, out.cpu().numpy())
    assert same and err < (1e-14 if prec == capi.FP64 else 1e-6), err
