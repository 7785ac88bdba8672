"""The FD-z column kernel over every x size it takes (8 and 16 points per
thread, one and two wavefronts per transform, one to 64 column pairs per
block) and over column counts that leave a pair or a block partly empty, all
jobs in one batch: FP64 against the oracle and against each job alone, FP32
against FP64.

Tolerance: a transform of N points is within 4 log2(N) units of rounding of
the exact one in norm (at most 5 operations per radix-2 level, random signs);
a product takes two inverse transforms and one forward, and its difference
along z multiplies the error by no more than the row's condition, nz^2 / 2 per
solve.  So FP64 states are held to 1e-12 + 12 nz^2 2^-53 and FP32 physical
fields, which are one transform away from the state, to 4 log2(nx) 2^-24 plus
the rounding of the velocities, which are stored in single precision."""
import numpy as np
import pytest

from conftest import rel
from oracle import melvin_oracle as O
from test_gpu_fdz import _job, _oracle_run, _rbc_start

pytestmark = pytest.mark.gpu

NX = [8, 16, 32, 64, 128, 256, 512, 1024, 2048]
NZ = [5, 6, 9, 24, 33, 130, 131]


def _cases():
    out = []
    for k, nx in enumerate(NX):
        for nz in NZ if nx <= 32 else (NZ[k % 3], NZ[3 + k % 4]):
            p = O.make_params(dict(nx=nx, nz=nz, lx=2.0, lz=1.0, Pr=1.0, Ra=1e5, alpha=0.51,
                                   integrator_order=2, spatial_derivative_order=2,
                                   discretisation=["spectral", "fdm"]))
            out.append((p, 1e-3 / nz ** 2) + tuple(_rbc_start(p, seed=40 + k)))
    return out


def _jobs(mlv, cases, dtype="f64"):
    jobs = []
    for p, dt, w0, t0 in cases:
        j = _job(mlv, p, "pc", dtype=dtype, dt=dt, want_phys=True)
        j.set_state([w0, t0])
        jobs.append(j)
    return jobs


def test_columns_vs_oracle_and_alone(mlv):
    cases = _cases()
    batch = _jobs(mlv, cases)
    b = mlv.fdz.FdzBatch(batch)
    b.step(3)
    b.step(1, write_phys=True)
    got = [(j.state(), j.physical()) for j in batch]
    b.close()
    for (p, dt, w0, t0), ((w, t), phys), j in zip(cases, got, _jobs(mlv, cases)):
        st = _oracle_run(p, O.step_rbc_pc, w0, t0, dt, 3)
        tol = 1e-12 + 12 * p.nz ** 2 * 2.0 ** -53
        for x, s in zip(phys[2:], (st["w"], st["tmp"])):
            assert rel(x, O.to_physical(p, s)) < tol, (p.nx, p.nz)
        O.step_rbc_pc(p, st)
        assert rel(w, st["w"]) < tol and rel(t, st["tmp"]) < tol, (p.nx, p.nz)
        b = mlv.fdz.FdzBatch([j])
        b.step(3)
        b.step(1, write_phys=True)
        for x, y in zip(j.state() + j.physical(), [w, t] + phys):
            np.testing.assert_array_equal(x, y)
        b.close()


def test_columns_single_precision(mlv):
    cases = _cases()
    out = []
    for dtype in ("f64", "f32"):
        jobs = _jobs(mlv, cases, dtype)
        b = mlv.fdz.FdzBatch(jobs)
        b.step(1, write_phys=True)
        out.append([(j.state(), j.physical()) for j in jobs])
        b.close()
    for (p, *_), (s64, p64), (s32, p32) in zip(cases, *out):
        tol = (4 * np.log2(p.nx) + 2) * 2.0 ** -24
        for x, y in zip(p32, p64):
            assert rel(x, y) < tol, (p.nx, p.nz)
        # a step's increments pass three transforms and stay below the state
        for x, y in zip(s32, s64):
            assert rel(x, y) < 3 * tol, (p.nx, p.nz)
