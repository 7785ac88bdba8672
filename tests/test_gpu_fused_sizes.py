"""The fused step at every grid extent from 8 to 4096 on either axis, against
the FP64 oracle, and the same bits whatever block sizes a batch takes (a
small batch runs smaller blocks than one that fills the device).

FP64: a step rounds each value a few dozen times relative to the fields it
is formed from, so 1e-12; FP32 with its compensated update, 1e-5."""
import numpy as np
import pytest

from conftest import rel
from oracle import melvin_oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (8, 512), (16, 4096), (32, 2048), (64, 16), (128, 1024), (256, 32), (512, 64),
         (1024, 8), (2048, 32), (4096, 16)]
FIELDS = {"vorticity": ("w",), "scalar": ("w", "c"), "ddc": ("w", "tmp", "xi"), "mhd": ("w", "j")}


def _problem(name, nx, nz, order):
    p = O.make_params(dict(nx=nx, nz=nz, lx=2.0, lz=1.5, initial_dt=1e-4,
                           spatial_derivative_order=order, Pr=7.0, R0=1.5, tau=0.01, Re=1e3, S=1e3))
    rng = np.random.default_rng(nx * 5 + nz)
    start = [O.to_spectral(p, rng.standard_normal((nx, nz))) for _ in FIELDS[name]]
    coeff = {"ddc": [7.0, 1.0, 0.01]}.get(name, [1e-3] * len(start))
    step = {"vorticity": lambda s: O.step_vorticity(p, s, 1e-3),
            "scalar": lambda s: O.step_vorticity(p, s, 1e-3, ("c",)),
            "ddc": lambda s: O.step_ddc(p, s), "mhd": lambda s: O.step_mhd(p, s)}[name]
    return p, start, coeff, step


def _job(mlv, name, p, start, coeff, dtype):
    j = mlv.fused.Job({"scalar": "vorticity"}.get(name, name), p.nx, p.nz, p.lx, p.lz, dtype=dtype,
                      dt=p.initial_dt, coeff=coeff, param=[7.0, 1.5] if name == "ddc" else (),
                      fd_order=p.spatial_derivative_order, want_phys=True)
    j.set_state(start)
    return j


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("name", sorted(FIELDS))
@pytest.mark.parametrize("nx,nz", SIZES)
def test_every_extent_vs_oracle(mlv, nx, nz, name, order):
    if nz == 4096 and name in ("ddc", "mhd"):
        pytest.skip("refused: the z pass of five or six channels does not fit 4096 points")
    p, start, coeff, step = _problem(name, nx, nz, order)
    st = O.new_state(p, FIELDS[name], dt=p.initial_dt)
    for f, s in zip(FIELDS[name], start):
        st[f] = s.copy()
    for _ in range(3):
        step(st)
    for dtype, tol in (("f64", 1e-12), ("f32", 1e-5)):
        job = _job(mlv, name, p, start, coeff, dtype)
        b = mlv.fused.Batch([job])
        b.step(3)
        for f, got in zip(FIELDS[name], job.state()):
            assert rel(got, st[f]) <= tol, (dtype, f)
        b.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", sorted(FIELDS))
@pytest.mark.parametrize("n", [64, 256, 512])
def test_same_bits_alone_and_filling_the_device(mlv, n, name, dtype):
    p, start, coeff, _ = _problem(name, n, n, 2)
    alone = _job(mlv, name, p, start, coeff, dtype)
    b = mlv.fused.Batch([alone])
    b.run_device(4, cadence=2)
    b.sync()
    want, track = alone.state(), b.tracker(0)
    b.close()
    many = [_job(mlv, name, p, start, coeff, dtype) for _ in range(48)]
    b = mlv.fused.Batch(many)
    b.run_device(4, cadence=2)
    b.sync()
    for k in (0, 31, 47):
        for x, y in zip(many[k].state(), want):
            np.testing.assert_array_equal(x, y)
        for key, v in b.tracker(k).items():
            np.testing.assert_array_equal(v, track[key])
    b.close()
