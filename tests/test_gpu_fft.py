"""GPU FFT passes against numpy.fft (a library routine) through the C ABI.

Shapes include extents of 256 along z or y, where a z or y pass block moves 16 pencils of 256
elements and its global loads run in two chunks of 8 per thread."""
import numpy as np
import pytest

import srx_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 16, 16), (4, 6, 10), (12, 20, 9), (32, 16, 64), (1, 8, 8),
                                   (8, 1, 5), (96, 8, 4), (4, 32, 256), (16, 256, 8)])
@pytest.mark.parametrize("ncomp", [1, 6, 9])
def test_forward_matches_numpy_fp64(shape, ncomp):
    rng = np.random.default_rng(hash((shape, ncomp)) % 2**32)
    x = rng.standard_normal((ncomp,) + shape)
    got = srx_amd.fft_forward(x)
    ref = np.fft.rfftn(x, axes=(1, 2, 3))
    assert got.shape == ref.shape
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err < 1e-13, err


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 16, 16), (12, 20, 9), (32, 16, 64), (96, 8, 4), (4, 32, 256),
                                   (16, 256, 8)])
def test_inverse_matches_numpy_fp64(shape):
    rng = np.random.default_rng(7)
    x = rng.standard_normal((9,) + shape)
    X = np.fft.rfftn(x, axes=(1, 2, 3))
    n = shape[0] * shape[1] * shape[2]
    got = srx_amd.fft_inverse(X, shape[2], scale=1.0 / n)
    assert np.abs(got - x).max() < 1e-13 * np.abs(x).max() * 10


def test_mixed_precision_forward_error_bound():
    rng = np.random.default_rng(3)
    x = rng.standard_normal((6, 32, 32, 32))
    got = srx_amd.fft_forward(x, precision=srx_amd.PREC_MIXED)
    ref = np.fft.rfftn(x, axes=(1, 2, 3))
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err < 5e-6, err


@pytest.mark.parametrize("prec", [srx_amd.PREC_FP64, srx_amd.PREC_MIXED])
@pytest.mark.parametrize("shape", [(1, 1, 1), (30, 3, 60), (32, 1, 64), (36, 2, 128), (64, 5, 2)])
def test_orders_of_the_spectrum_at_tile_edges(shape, prec):
    """The entry points turn spectra around in 32 x 32 pieces of x and kz: both directions at extents
    around one and two pieces, with the FP64 bounds of the tests above and log2(N) roundings of 2^-23
    of the largest value in mixed precision."""
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((2,) + shape)
    X = np.fft.rfftn(x, axes=(1, 2, 3))
    tol = 1e-13 if prec == srx_amd.PREC_FP64 else 20 * 2.0**-23
    got = srx_amd.fft_forward(x, precision=prec)
    assert np.abs(got - X).max() <= tol * np.abs(X).max()
    back = srx_amd.fft_inverse(X, shape[2], precision=prec, scale=1.0 / np.prod(shape))
    assert np.abs(back - x).max() <= 10 * tol * np.abs(x).max()
