"""Transforms of many short rows, whose blocks take up to 128 rows through LDS
at once from 65536 rows on: row counts around a block's and around that limit,
every short length and the first one beyond, both directions, against
numpy.fft; and the x passes' block widths on either side of their limit.  Bounds as for the other
transforms: FP64 1e-13, FP32 2e-6 relative L2."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-13, np.float32: 2e-6}


def _check(mlv, name, a, want, dtype, **kw):
    out = getattr(mlv.hip.fft, name)(mlv.hip.asarray(a), **kw).cpu().numpy()
    assert out.shape == want.shape
    assert rel(out, want) <= TOL[dtype]


def _spectrum(rng, shape, dtype):
    c = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    return c.astype(np.complex128 if dtype == np.float64 else np.complex64)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [8, 16, 32, 64])
@pytest.mark.parametrize("rows", [1, 2, 3, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1000, 65535, 65536, 65537,
                                  65567, 65663])
def test_short_rows(mlv, rows, n, dtype):
    rng = np.random.default_rng(rows + n)
    a = rng.standard_normal((rows, n)).astype(dtype)
    _check(mlv, "rfft", a, np.fft.rfft(a.astype(np.float64), axis=1), dtype, axis=1)
    c = _spectrum(rng, (rows, n // 2 + 1), dtype)
    _check(mlv, "irfft", c, np.fft.irfft(c.astype(np.complex128), axis=1), dtype, axis=1)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(8, 8), (128, 8), (512, 16), (4096, 8), (64, 32)])
def test_short_rows_of_two_dimensions(mlv, shape, dtype):
    rng = np.random.default_rng(sum(shape))
    a = rng.standard_normal(shape).astype(dtype)
    _check(mlv, "rfft2", a, np.fft.rfft2(a.astype(np.float64)), dtype)
    c = _spectrum(rng, (shape[0], shape[1] // 2 + 1), dtype)
    _check(mlv, "irfft2", c, np.fft.irfft2(c.astype(np.complex128)), dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [8, 64, 256, 1024, 2048])
@pytest.mark.parametrize("cols", [2045, 2046, 2047, 2049, 8191])
def test_many_columns(mlv, cols, n, dtype):
    rng = np.random.default_rng(cols + n)
    a = rng.standard_normal((n, cols)).astype(dtype)
    _check(mlv, "rfft", a, np.fft.rfft(a.astype(np.float64), axis=0), dtype, axis=0)
    c = _spectrum(rng, (n // 2 + 1, cols), dtype)
    _check(mlv, "irfft", c, np.fft.irfft(c.astype(np.complex128), axis=0), dtype, axis=0)
