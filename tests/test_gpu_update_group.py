"""The single-precision update in blocks of a whole column group (shape 2, x
sizes of 512 and 1024) gives the other shapes' bits: column counts that fill
their last group and that do not, both orders, every problem, with and without
the carry, several jobs of different z sizes; and the shapes that a batch
starts with."""
import ctypes

import numpy as np
import pytest

from test_gpu_fused_sizes import FIELDS, _job, _problem

pytestmark = pytest.mark.gpu


def _run(mlv, jobs, update, steps=5):
    b = mlv.fused.Batch(jobs)
    b.set_plan(0, 0, update)
    b.run_device(steps, cadence=2)
    b.sync()
    out = [j.state() for j in jobs]
    tr = [b.tracker(k) for k in range(len(jobs))]
    b.close()
    return out, tr


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("name", sorted(FIELDS))
@pytest.mark.parametrize("nx,nz", [(512, 8), (512, 32), (512, 128), (1024, 16), (1024, 64),
                                   (1024, 1024)])
def test_group_update_gives_the_same_bits(mlv, nx, nz, name, order):
    p, start, coeff, _ = _problem(name, nx, nz, order)
    want, track = _run(mlv, [_job(mlv, name, p, start, coeff, "f32")], 0)
    for update in (1, 2):
        got, tr = _run(mlv, [_job(mlv, name, p, start, coeff, "f32")], update)
        for a, b in zip(got[0], want[0]):
            assert np.isfinite(a).all()
            np.testing.assert_array_equal(a, b)
        for k, v in tr[0].items():
            np.testing.assert_array_equal(v, track[0][k])


@pytest.mark.parametrize("compensated", [True, False])
@pytest.mark.parametrize("ab", [2, 4])
def test_group_update_of_mixed_z_sizes(mlv, ab, compensated):
    def jobs():
        out = []
        for nz in (8, 64, 256):
            p, start, _, _ = _problem("scalar", 512, nz, 2)
            j = mlv.fused.Job("vorticity", 512, nz, p.lx, p.lz, dtype="f32", dt=1e-4,
                              coeff=[1e-3, 1e-3], ab_order=ab, compensated=compensated)
            j.set_state(start)
            out.append(j)
        return out

    want, _ = _run(mlv, jobs(), 0, 7)
    got, _ = _run(mlv, jobs(), 2, 7)
    for a, b in zip(got, want):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)


def _default_plan(mlv, sizes, problem="vorticity", coeff=(1e-3, 1e-3)):
    jobs = [mlv.fused.Job(problem, n, n, 2.0, 2.0, dtype="f32", coeff=coeff, param=[7.0, 1.5])
            for n in sizes]
    b = mlv.fused.Batch(jobs)
    p = (ctypes.c_int * 7)()
    mlv._lib.call("mlv_batch_plan", b.handle, p)
    b.close()
    return p[0], p[2]


def test_default_shapes(mlv):
    """(x-inverse, update): one column a block is not taken, nor the smaller
    x-inverse block on a large launch of partial lines."""
    ddc = dict(problem="ddc", coeff=(7.0, 1.0, 0.01))
    assert _default_plan(mlv, [512]) == (0, 0)
    assert _default_plan(mlv, [1024]) == (0, 0)
    assert _default_plan(mlv, [2048, 256, 512, 256]) == (1, 0)
    assert _default_plan(mlv, [256] * 64) == (1, 0)
    assert _default_plan(mlv, [512] * 64, **ddc) == (0, 2)
    assert _default_plan(mlv, [1024] * 16) == (0, 2)
