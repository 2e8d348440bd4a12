"""E-basis, laboratory frame, FP32: an angle's intensity where the quadratic form's terms
cancel.

One material aligned along (1, 1, 0) with n_perp = 1: N = d w s s^T, so the intensity of E at
angle theta goes with (cos theta + sin theta)^2.  The eleven angles 134.8 ... 135.2 degrees
average to 8e-6 of the form's components: components rounded to FP32 (6e-8) leave about
7e-3 of the average, projections of each angle about 3e-5, FP64 forms of the same fields
less.  Bar as in every FP32 parity test, 1e-4 of the FP64 oracle.
"""
import numpy as np
import pytest

from cyrsoxs_amd import capi, synthetic
from oracle import oracle as O
from tests.helpers import pattern_rel_l2

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(64, 64, 16), (48, 50, 12), (64, 64, 1), (40, 36, 1)])
def test_cancelling_forms(dims):
    print(f"cancelling forms {dims}", flush=True)
    V = dims[0] * dims[1] * dims[2]
    w = np.random.default_rng(3).uniform(0.2, 1.0, V).astype(np.float32)
    vox = np.zeros((1, V, 4))
    vox[0, :, 0] = vox[0, :, 1] = w
    mats = np.array([[[1 - 1e-3, 1e-3, 1.0, 0.0]], [[1 - 2e-3, 5e-4, 1.0, 0.0]]])
    args = (dims, 1, 2.0, [284.0, 287.0], (134.8, 0.04, 135.2))
    kw = dict(interpolation=1, windowing=1, morphology_type=1)
    ref = O.simulate(O.Sim(*args, **kw), vox, mats)
    sim = capi.Sim(*args, pipeline=capi.PIPE_EBASIS, **kw)
    assert sim.num_angles == 11 and sim.resolved_pipeline() == capi.PIPE_EBASIS
    err, same = pattern_rel_l2(capi.simulate(sim, vox, mats), ref)
    assert same and err < 1e-4, (dims, err)


@pytest.mark.gpu
@pytest.mark.parametrize("rot_mask", [0, 1])
@pytest.mark.parametrize("n", [64, 256])
def test_whole_turns_of_large_values(n, rot_mask):
    """Whole turns of FP32 forms whose sum over the quarter turns exceeds FP32's largest value
    (3.4e38) while each is below it (four Bragg peaks of 2e38, 90 degrees apart): FP32 against
    FP64, 1e-4 as above."""
    print(f"large values {n} mask={rot_mask}", flush=True)
    dims, V = (n, n, 1), n * n
    a = 2 * np.pi * 8 * np.arange(n) / n
    vox = np.zeros((1, V, 4))
    vox[0, :, 3] = (2 + np.cos(a)[:, None] + np.cos(a)[None, :]).reshape(V)
    mats = np.array([[[1 - 2e-3, 1e-3, 1 - 1e-3, 5e-4]]])
    kw = dict(interpolation=1, morphology_type=1, rot_mask=rot_mask, pipeline=capi.PIPE_MBASIS)
    one = capi.simulate(capi.Sim(dims, 1, 1.0, [285.0], (0, 1, 0), precision=capi.FP64, **kw), vox, mats)
    vox *= np.sqrt(2e38 / np.nanmax(one))
    args = (dims, 1, 1.0, [285.0], (0.0, 2.0, 358.0))
    ref = capi.simulate(capi.Sim(*args, precision=capi.FP64, **kw), vox, mats)
    got = capi.simulate(capi.Sim(*args, **kw), vox, mats).astype(np.float64)
    err, same = pattern_rel_l2(got / 1e38, ref / 1e38)
    assert same and err < 1e-4, (n, rot_mask, err)


def _smooth(shape, seed):
    f = torch.randn(shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    return synthetic.gaussian_filter_periodic(f, 3.0).reshape(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,angles", [((40, 44, 12), (0.0, 10.0, 170.0)), ((100, 100, 20), (0.0, 1.0, 0.0))])
def test_few_forms_of_the_material_basis(dims, angles):
    """Small grids in FP32: the material basis, which AUTO takes for time, leaves no more than
    the per-angle executor.  Both errors (against FP64) are sums of a few roundings at the
    brightest pixels, about 25 % apart from seed to seed when averaged over eight, so their
    ratio stays below 1 + sqrt(2) x 0.25 = 1.35 (FP32 combinations and forms: 1.6)."""
    M, energies, err = 3, [281.0, 284.0, 286.0, 289.0], {}
    for seed in range(8):
        nx, ny, nz = dims
        logits = torch.stack([_smooth((nz, ny, nx), 100 * seed + m) for m in range(M)])
        logits = (logits - logits.mean(1, keepdim=True)) / logits.std(1, keepdim=True)
        phi = torch.softmax(logits, 0).numpy()
        rng = np.random.default_rng(seed)
        d = rng.normal(size=(M, phi.shape[1], 3))
        d /= np.linalg.norm(d, axis=-1, keepdims=True)
        s = rng.uniform(0, 1, size=phi.shape)
        vox = np.concatenate([d * np.sqrt(phi * s)[..., None], (phi * (1 - s))[..., None]], -1).astype(np.float32)
        mats = synthetic.lorentzian_constants(energies, M, seed=seed)
        kw = dict(interpolation=1, morphology_type=1)
        run = lambda prec, pipe: capi.simulate(capi.Sim(dims, M, 2.0, energies, angles, precision=prec, pipeline=pipe, **kw),
                                               vox, mats)
        ref = run(capi.FP64, capi.PIPE_PLAIN)
        for pipe in (capi.PIPE_PLAIN, capi.PIPE_MBASIS):
            err.setdefault(pipe, []).append(pattern_rel_l2(run(capi.FP32, pipe), ref)[0])
    rms = {p: float(np.sqrt(np.mean(np.square(e)))) for p, e in err.items()}
    print(rms)
    assert rms[capi.PIPE_MBASIS] < 1.35 * rms[capi.PIPE_PLAIN], rms
