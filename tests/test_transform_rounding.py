"""Rounding errors of single-axis transforms without a codelet, against extended precision.

FP32, sides below 208 that need a convolution: the arithmetic is FP64, so an output's error
is its own rounding, at most 2^-24 = 6e-8 of it, also where the pencil has a large mean.
FP64: up to eleven steps (2 x 4 stages, three products), each about 0.8 x 2^-53 rms, times
sqrt(m / n) <= 1.75 for a convolution's longer pencil: sqrt(11) x 0.8 x 1.1e-16 x 1.75 = 5.1e-16,
6e-16 with a margin.  Tables rounded from double arithmetic alone would add up to 4e-16 an
entry (the argument 2 pi k / n is that far off).
"""
import numpy as np
import pytest
import scipy.fft

from cyrsoxs_amd import capi

torch = pytest.importorskip("torch")


def _axis(x, axis, prec):
    """x: [n_rows, n] (axis 0: along rows) or [n, columns] (axis 1)."""
    d = torch.from_numpy(x.copy()).cuda()
    capi.fft_axis_device([d], (x.shape[1], x.shape[0], 1), prec, axis)
    torch.cuda.synchronize()
    ref = scipy.fft.fft(x.astype(np.clongdouble), axis=1 if axis == 0 else 0)
    return d.cpu().numpy().astype(np.clongdouble), ref


def _rel(a, b):
    return float(np.sqrt((abs(a - b) ** 2).sum() / (abs(b) ** 2).sum()))


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("n", [17, 23, 31, 34, 47, 61, 94, 101, 127, 155, 202])
def test_short_fp32_convolutions(n, axis):
    rng = np.random.default_rng(n)
    x = 1 + 0.1 * rng.normal(size=(n, 600)) + 0.1j * rng.normal(size=(n, 600))
    x = (x if axis else x.T).astype(np.complex64)
    got, ref = _axis(np.ascontiguousarray(x), axis, capi.FP32)
    off = np.s_[1:] if axis else np.s_[:, 1:]  # the values beside the mean's
    assert _rel(got[off], ref[off]) < 6e-8
    assert _rel(got, ref) < 6e-8


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("n", [13, 22, 33, 47, 61, 85, 101, 119, 200, 240])
def test_fp64_tables(n, axis):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 600)) + 1j * rng.normal(size=(n, 600))
    got, ref = _axis(np.ascontiguousarray(x if axis else x.T), axis, capi.FP64)
    assert _rel(got, ref) < 6e-16
