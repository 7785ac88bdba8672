"""Long axes whose calls run as separate operators: the result is theirs bit
for bit.  (The fused forms round otherwise.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fdz(mlv, nx, nz, precision, order):
    p = mlv.Parameters(dict(nx=nx, nz=nz, lx=2.0, lz=1.5, final_time=1.0, precision=precision,
                            spatial_derivative_order=order, integrator="explicit",
                            discretisation=["spectral", "fdm"]))
    sim = mlv.Simulation(p, mlv.hip)
    bfs = [mlv.BasisFunctions.COMPLEX_EXP, mlv.BasisFunctions.FDM]
    rng = np.random.default_rng(nx + nz)
    s = rng.standard_normal(p.spectral_shape) + 1j * rng.standard_normal(p.spectral_shape)
    return p, sim, bfs, mlv.hip.asarray(s.astype(p.complex))


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("nx,nz", [(2048, 64), (4096, 7), (4096, 64)])
def test_fdz_advection_beyond_1024_points(mlv, nx, nz, order, precision):
    import torch

    p, sim, bfs, s = _fdz(mlv, nx, nz, precision, order)
    a, b = (sim.make_variable("v", bfs) for _ in range(2))
    a.sets(s)
    b.sets(s)
    rng = np.random.default_rng(3)
    ux, uz = (mlv.hip.asarray(rng.standard_normal((nx, nz)).astype(p.float)) for _ in range(2))
    want = b.vec_dot_nabla(ux, uz, out=torch.empty_like(b.getp()))
    assert torch.equal(a.vec_dot_nabla(ux, uz), want)
    assert torch.equal(a.getp(), b.getp())


@pytest.mark.parametrize("precision", ["double", "single"])
def test_velocity_of_rows_beyond_a_block(mlv, precision):
    import torch

    p, sim, bfs, s = _fdz(mlv, 32, 4099, precision, 2)
    w, psi, ux, uz = (sim.make_variable(n, bfs) for n in ("w", "psi", "ux", "uz"))
    w.sets(s)
    sim.init_laplacian_solver(bfs)
    mlv.utility.calc_velocity_from_vorticity(w, psi, ux, uz, sim.get_laplacian_solver())
    assert torch.equal(psi.gets(), sim.get_laplacian_solver().solve(-w.gets()))
    assert torch.equal(uz.gets(), psi.sddx())
    assert torch.equal(ux.getp(), -psi.pddz())


def test_flux_of_the_advection_is_an_array_of_its_own(mlv):
    import torch
    from melvin_amd import _lib
    from melvin_amd._plans import plan_for, ptr

    p, sim, bfs, s = _fdz(mlv, 64, 17, "double", 2)
    pl = plan_for(p)
    f, ux, uz, flux = (torch.ones((64, 17), device="cuda", dtype=torch.float64) for _ in range(4))
    spec = torch.empty((pl.rows, pl.cols), device="cuda", dtype=pl.cplx)
    for bad in (f, ux, uz):
        with pytest.raises(ValueError, match="flux_phys"):
            _lib.call("mlv_advect_stencil", pl.handle, ptr(ux), ptr(uz), ptr(s), ptr(f), ptr(bad),
                      ptr(spec), _lib.stream_handle())
    _lib.call("mlv_advect_stencil", pl.handle, ptr(ux), ptr(uz), ptr(s), ptr(f), ptr(flux),
              ptr(spec), _lib.stream_handle())
    want = torch.empty_like(spec)
    _lib.call("mlv_advect", pl.handle, ptr(ux), ptr(uz), ptr(s), ptr(f), ptr(want),
              _lib.stream_handle())
    assert torch.allclose(spec, want, rtol=0, atol=1e-12 * float(want.abs().max()))
