"""The FD-z row kernel at the row lengths where its split changes: the last nz
of each chunk length, the first of the next and the shortest and longest rows,
all in one launch, against the oracle and against each job alone.

Tolerance: the row solves are backward stable with a condition number of at
most nz^2 / 2 and each step passes through two of them, so six FP64 steps stay
within 12 nz^2 units of rounding of the oracle's, beside the 1e-12 of the
transforms; the same bits alone."""
import numpy as np
import pytest

from conftest import rel
from oracle import melvin_oracle as O
from test_gpu_fdz import _job, _oracle_run, _rbc_start

pytestmark = pytest.mark.gpu

NZ = [7, 64, 65, 128, 129, 256, 257, 512, 513, 767, 768]


@pytest.mark.parametrize("scheme,order,ab", [("pc", 2, 2), ("semi-implicit", 2, 4),
                                             ("explicit", 4, 2)])
def test_row_splits_in_one_launch(mlv, scheme, order, ab):
    step = {"pc": "step_rbc_pc", "semi-implicit": "step_rbc_semi_implicit",
            "explicit": "step_rbc"}[scheme]
    cases = []
    for k, nz in enumerate(NZ):
        p = O.make_params(dict(nx=16 << (k % 2), nz=nz, lx=2.0, lz=1.0, Pr=1.0, Ra=1e5,
                               alpha=0.51, integrator_order=ab, spatial_derivative_order=order,
                               discretisation=["spectral", "fdm"]))
        cases.append((p, 1e-3 / nz ** 2) + tuple(_rbc_start(p, seed=20 + k)))

    def jobs():
        out = []
        for p, dt, w0, t0 in cases:
            j = _job(mlv, p, scheme, dt=dt)
            j.set_state([w0, t0])
            out.append(j)
        return out

    batch = jobs()
    b = mlv.fdz.FdzBatch(batch)
    b.step(6)
    got = [j.state() for j in batch]
    b.close()
    for (p, dt, w0, t0), (w, t), j in zip(cases, got, jobs()):
        st = _oracle_run(p, getattr(O, step), w0, t0, dt, 6)
        tol = 1e-12 + 12 * p.nz ** 2 * 2.0 ** -53
        assert rel(w, st["w"]) < tol and rel(t, st["tmp"]) < tol, p.nz
        b = mlv.fdz.FdzBatch([j])
        b.step(6)
        for x, y in zip(j.state(), (w, t)):
            np.testing.assert_array_equal(x, y)
        b.close()
