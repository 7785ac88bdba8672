"""The advection and velocity calls that form their input inside a transform
against the separate operators (stencil kernel, then transform), which they
replace: edges of the transform splits, odd FD-z extents, both orders.

Both round each product, difference and transform a few times; the largest
term is a product over a grid spacing, so the difference of two spectra is
bounded by a few tens of units of rounding times that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = {"double": 2.0 ** -53, "single": 2.0 ** -24}
FULL = [(8, 8), (16, 1024), (64, 32), (128, 4096), (512, 256), (1024, 64), (2048, 16), (4096, 8)]
FDZ = [(8, 5), (16, 9), (64, 33), (256, 130), (1024, 17), (2048, 6), (4096, 7), (32, 700)]


def _make(mlv, nx, nz, fdz, precision, order):
    p = mlv.Parameters(dict(nx=nx, nz=nz, lx=2.0, lz=1.5, final_time=1.0, precision=precision,
                            spatial_derivative_order=order, integrator="explicit" if fdz else
                            "semi-implicit", discretisation=["spectral", "fdm" if fdz else "spectral"]))
    sim = mlv.Simulation(p, mlv.hip)
    B = mlv.BasisFunctions
    bfs = [B.COMPLEX_EXP, B.FDM if fdz else B.COMPLEX_EXP]
    return p, sim, bfs


def _random_spectrum(mlv, p, seed):
    rng = np.random.default_rng(seed)
    shape = p.spectral_shape
    return mlv.hip.asarray((rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
                           .astype(p.complex))


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("nx,nz,fdz", [s + (False,) for s in FULL] + [s + (True,) for s in FDZ])
def test_advect_equals_stencil_then_transform(mlv, nx, nz, fdz, order, precision):
    import torch

    p, sim, bfs = _make(mlv, nx, nz, fdz, precision, order)
    rng = np.random.default_rng(nx + nz)
    ux, uz = (mlv.hip.asarray(rng.standard_normal((nx, nz)).astype(p.float)) for _ in range(2))
    a, b = (sim.make_variable("v", bfs) for _ in range(2))
    s = _random_spectrum(mlv, p, 1)
    a.sets(s)
    b.sets(s)
    got = a.vec_dot_nabla(ux, uz)
    want = b.vec_dot_nabla(ux, uz, out=torch.empty_like(b.getp()))
    assert torch.equal(a.getp(), b.getp())
    top = float((a.getp().abs().max() * max(ux.abs().max(), uz.abs().max())).item())
    bound = 40 * EPS[precision] * top * (1 / p.dx + 1 / p.dz)
    assert float((got - want).abs().max()) <= bound
    # without the conversion: the physical field as it stands
    got2 = a.vec_dot_nabla(ux, uz, convert_to_physical=False)
    assert torch.equal(got2, got)


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("nx,nz,fdz", [s + (False,) for s in FULL] + [s + (True,) for s in FDZ])
def test_velocity_equals_separate_operators(mlv, nx, nz, fdz, precision):
    import torch

    p, sim, bfs = _make(mlv, nx, nz, fdz, precision, 2)
    w, psi, ux, uz = (sim.make_variable(n, bfs) for n in ("w", "psi", "ux", "uz"))
    w.sets(_random_spectrum(mlv, p, 2))
    sim.init_laplacian_solver(bfs)
    mlv.utility.calc_velocity_from_vorticity(w, psi, ux, uz, sim.get_laplacian_solver())
    ref = sim.get_laplacian_solver().solve(-w.gets())
    kx = mlv.hip.asarray(2 * np.pi / p.lx * sim._array_factory.make_mode_number_matrices()[0].cpu().numpy())
    eps = EPS[precision]
    scale = float(ref.abs().max())
    assert float((psi.gets() - ref).abs().max()) <= 4 * eps * scale
    assert (float((uz.gets() - 1j * kx * ref).abs().max())
            <= 8 * eps * float((kx * ref).abs().max()))
    st = sim._spectral_trans
    assert torch.equal(uz.getp(), st.to_physical(uz.gets(), basis_functions=bfs))
    if fdz:
        assert torch.equal(psi.getp(), st.to_physical(psi.gets(), basis_functions=bfs))
        assert torch.equal(ux.getp(), -psi.pddz())
    else:
        assert torch.equal(ux.getp(), st.to_physical(ux.gets(), basis_functions=bfs))
    assert torch.isfinite(ux.getp()).all()


@pytest.mark.parametrize("fdz", [False, True])
def test_velocity_arguments_that_share_the_fields_memory(mlv, fdz):
    """The field's own physical array as a velocity, as it is and transposed
    (a view that has to be copied after the conversion, not before)."""
    import torch

    p, sim, bfs = _make(mlv, 64, 64, fdz, "double", 2)
    for view in (lambda v: v.getp(), lambda v: v.getp().T):
        a, b = (sim.make_variable("v", bfs) for _ in range(2))
        for v in (a, b):
            v.sets(_random_spectrum(mlv, p, 3))
            v.getp().fill_(7.0)
        got = a.vec_dot_nabla(view(a), view(a))
        want = b.vec_dot_nabla(view(b), view(b), out=torch.empty_like(b.getp()))
        top = float(a.getp().abs().max()) ** 2
        bound = 40 * EPS["double"] * top * (1 / p.dx + 1 / p.dz)
        assert float((got - want).abs().max()) <= bound


def test_overridden_transforms_are_used(mlv):
    """A transformer or variable class of the caller's own keeps its say."""
    p, sim, bfs = _make(mlv, 32, 32, False, "double", 2)

    class Doubling(mlv.SpectralTransformer):
        def to_spectral(self, *a, **k):
            return 2.0 * super().to_spectral(*a, **k)

    ux, uz = (mlv.hip.asarray(np.random.default_rng(k).standard_normal((32, 32))) for k in (1, 2))
    a, b = (sim.make_variable("v", bfs) for _ in range(2))
    for v in (a, b):
        v.sets(_random_spectrum(mlv, p, 4))
    b._st = Doubling(p, mlv.hip)
    got, want = a.vec_dot_nabla(ux, uz), b.vec_dot_nabla(ux, uz)
    scale = float(want.abs().max())
    assert float((2.0 * got - want).abs().max()) <= 1e-10 * scale
