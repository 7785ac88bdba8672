"""Methods that a caller's own class or instance puts in place of this
package's are used by the calls that otherwise form several of them in one
launch: calc_velocity_from_vorticity and vec_dot_nabla.

Each replacement doubles what it returns (or takes), so the call's results
are exact multiples of the plain ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fields(mlv, fdz, order, n=4):
    p = mlv.Parameters(dict(nx=64, nz=33 if fdz else 32, lx=2.0, lz=1.5, final_time=1.0,
                            precision="double", spatial_derivative_order=order,
                            integrator="explicit" if fdz else "semi-implicit",
                            discretisation=["spectral", "fdm" if fdz else "spectral"]))
    sim = mlv.Simulation(p, mlv.hip)
    B = mlv.BasisFunctions
    bfs = [B.COMPLEX_EXP, B.FDM if fdz else B.COMPLEX_EXP]
    var = [sim.make_variable(f"v{k}", bfs) for k in range(n)]
    rng = np.random.default_rng(11)
    s = rng.standard_normal(p.spectral_shape) + 1j * rng.standard_normal(p.spectral_shape)
    var[0].sets(mlv.hip.asarray(s))
    sim.init_laplacian_solver(bfs)
    return p, sim, var


def _velocity(mlv, fdz, order, change=lambda mlv, p, w, psi, ux, uz: None):
    p, sim, (w, psi, ux, uz) = _fields(mlv, fdz, order)
    change(mlv, p, w, psi, ux, uz)
    mlv.utility.calc_velocity_from_vorticity(w, psi, ux, uz, sim.get_laplacian_solver())
    return ux._pdata.clone(), uz._pdata.clone()


def _class_method(name):
    """The streamfunction in a subclass whose method returns twice as much."""
    def change(mlv, p, w, psi, ux, uz):
        base = type(psi)

        class Twice(base):
            pass

        setattr(Twice, name, lambda self: 2.0 * getattr(base, name)(self))
        psi.__class__ = Twice
    return change


def _instance_pddz(mlv, p, w, psi, ux, uz):
    plain = psi.pddz
    psi.pddz = lambda: 2.0 * plain()


def _class_setp(mlv, p, w, psi, ux, uz):
    base = type(ux)

    class Twice(base):
        def setp(self, data):
            super().setp(2.0 * data)

    ux.__class__ = Twice


def _own_differentiator(mlv, p, w, psi, ux, uz):
    class Twice(mlv.SpatialDifferentiator):
        def pddz(self, var, out=None):
            return 2.0 * super().pddz(var, out)

    psi._sd = Twice(p, mlv.hip)


def _instance_differentiator(mlv, p, w, psi, ux, uz):
    psi._sd = mlv.SpatialDifferentiator(p, mlv.hip)
    plain = psi._sd.pddz
    psi._sd.pddz = lambda var, out=None: 2.0 * plain(var, out)


def _other_order(mlv, p, w, psi, ux, uz):
    """A differentiator of the other order."""
    q = mlv.Parameters(dict(nx=p.nx, nz=p.nz, lx=p.lx, lz=p.lz, final_time=1.0, precision="double",
                            spatial_derivative_order=6 - p.spatial_derivative_order,
                            integrator="explicit", discretisation=["spectral", "fdm"]))
    psi._sd = mlv.SpatialDifferentiator(q, mlv.hip)


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("change", [
    _class_method("pddz"), _class_method("getp"), _instance_pddz, _class_setp, _own_differentiator,
    _instance_differentiator],
    ids=["class pddz", "class getp", "instance pddz", "class setp", "class sd", "instance sd"])
def test_fdz_velocity_uses_the_callers_methods(mlv, change, order):
    import torch

    ux, uz = _velocity(mlv, True, order)
    gx, gz = _velocity(mlv, True, order, change)
    assert torch.equal(gx, 2.0 * ux)
    assert torch.equal(gz, uz)


def test_fdz_velocity_uses_a_differentiator_of_another_order(mlv):
    import torch

    for order in (2, 4):
        want = _velocity(mlv, True, 6 - order)[0]
        assert torch.equal(_velocity(mlv, True, order, _other_order)[0], want)


@pytest.mark.parametrize("how", ["class", "instance", "transformer"])
@pytest.mark.parametrize("fdz", [False, True])
def test_velocity_uses_the_callers_transforms(mlv, fdz, how):
    import torch

    def change(mlv, p, w, psi, ux, uz):
        if how == "class":
            base = type(uz)

            class Twice(base):
                def to_physical(self):
                    super().to_physical()
                    self._pdata.mul_(2.0)

            uz.__class__ = Twice
        else:
            uz._st = mlv.SpectralTransformer(p, mlv.hip)
            target = uz if how == "instance" else uz._st
            plain = target.to_physical

            def twice(*a, **k):
                plain(*a, **k)
                uz._pdata.mul_(2.0)

            target.to_physical = twice

    ux, uz = _velocity(mlv, fdz, 2)
    gx, gz = _velocity(mlv, fdz, 2, change)
    assert torch.equal(gx, ux)
    assert torch.equal(gz, 2.0 * uz)


@pytest.mark.parametrize("order", [2, 4])
def test_fdz_velocity_is_the_separate_operators(mlv, order):
    """Both orders of the z difference that the one call forms itself."""
    import torch

    p, sim, (w, psi, ux, uz) = _fields(mlv, True, order)
    mlv.utility.calc_velocity_from_vorticity(w, psi, ux, uz, sim.get_laplacian_solver())
    assert torch.equal(ux.getp(), -psi.pddz())
    assert float(ux.getp().abs().max()) > 0.0


def test_advection_uses_the_callers_transform_of_an_instance(mlv):
    import torch

    p, sim, (a, b) = _fields(mlv, False, 2, 2)
    b.sets(a.gets())
    b._st = mlv.SpectralTransformer(p, mlv.hip)
    plain = b._st.to_spectral
    b._st.to_spectral = lambda *x, **k: 2.0 * plain(*x, **k)
    ux, uz = (mlv.hip.asarray(np.random.default_rng(k).standard_normal((p.nx, p.nz)))
              for k in (1, 2))
    want = 2.0 * a.vec_dot_nabla(ux, uz)
    got = b.vec_dot_nabla(ux, uz)
    # one forms the flux inside the transform: a few dozen roundings of its terms
    top = float(a.getp().abs().max() * max(ux.abs().max(), uz.abs().max()))
    assert float((got - want).abs().max()) <= 80 * 2.0 ** -53 * top * (1 / p.dx + 1 / p.dz)
