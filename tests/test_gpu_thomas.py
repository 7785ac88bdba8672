"""The FD-z Poisson solve at the row lengths where its work split changes:
the last row of each block size, the first of the next, the longest row a
block holds and the first one beyond it, and the shortest rows.

Reference: Thomas's sweep in FP64 NumPy.  Both are backward stable for this
M-matrix, whose condition number is at most nz^2 / 2 (the kx = 0 mode), so
they agree within a few units of rounding times that."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sweep(rhs, lx, dz):
    nn, nz = rhs.shape
    k = 2.0 * np.pi / lx * np.arange(nn)
    lo, dg = 1.0 / dz ** 2, -(k ** 2 + 2.0 / dz ** 2)
    c, d = np.zeros((nn, nz)), rhs.copy()
    for j in range(1, nz - 1):
        r = 1.0 / (dg - lo * c[:, j - 1])
        c[:, j] = lo * r
        d[:, j] = (rhs[:, j] - lo * d[:, j - 1]) * r
    for j in range(nz - 2, 0, -1):
        d[:, j] -= c[:, j] * d[:, j + 1]
    return d


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("nz", [5, 6, 64, 65, 255, 256, 257, 512, 513, 1025, 2047, 2049, 4096, 4097])
def test_solve_at_the_edges_of_the_split(mlv, nz, precision):
    import torch

    p = mlv.Parameters(dict(nx=32, nz=nz, lx=2.0, lz=1.0, final_time=1.0, precision=precision,
                            integrator="explicit", discretisation=["spectral", "fdm"]))
    B = mlv.BasisFunctions
    ls = mlv.LaplacianSolver(p, mlv.hip, [B.COMPLEX_EXP, B.FDM])
    rng = np.random.default_rng(nz)
    rhs = rng.standard_normal((p.nn, nz)) + 1j * rng.standard_normal((p.nn, nz))
    rhs = rhs.astype(p.complex).astype(np.complex128)
    want = _sweep(rhs, p.lx, p.dz)
    eps = 2.0 ** -53
    tol = 4 * nz ** 2 * eps + (0 if precision == "double" else 2.0 ** -23)
    src = mlv.hip.asarray(rhs.astype(p.complex))
    got = ls.solve(src).cpu().numpy()
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    # psi = solve(-w) and uz = i kx psi in one call, psi overwriting w
    uz = torch.empty_like(src)
    L = mlv._lib
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L.call("mlv_velocity", ls._plan.handle, ptr(src), ptr(src), ctypes.c_void_p(0), ptr(uz),
           L.stream_handle())
    psi = src.cpu().numpy()
    assert np.array_equal(psi, -got)
    kx = 2.0 * np.pi / p.lx * np.arange(p.nn)[:, None]
    rel = 2.0 ** -52 if precision == "double" else 2.0 ** -23
    assert np.abs(uz.cpu().numpy() - 1j * kx * psi).max() <= rel * np.abs(kx * psi).max()
