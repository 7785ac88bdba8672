"""Double precision at the lengths where a kernel or its compiled size
changes: each z-pass plan and each block shape of the x passes at 1024, 2048
and 4096 points against the FP64 oracle, and the shapes against each other
bit for bit.  (A step rounds each value a few dozen times: 1e-12.)"""
import itertools

import numpy as np
import pytest

from conftest import rel
from oracle import melvin_oracle as O
from test_gpu_fused_sizes import FIELDS, _job, _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(FIELDS))
@pytest.mark.parametrize("nx,nz", [(16, 1024), (16, 2048), (64, 4096), (1024, 16), (2048, 16),
                                   (4096, 16), (2048, 2048)])
def test_every_plan_vs_oracle(mlv, nx, nz, name):
    if nz == 4096 and name in ("ddc", "mhd"):
        pytest.skip("refused: the z pass of five or six channels does not fit 4096 points")
    p, start, coeff, step = _problem(name, nx, nz, 4)
    st = O.new_state(p, FIELDS[name], dt=p.initial_dt)
    for f, s in zip(FIELDS[name], start):
        st[f] = s.copy()
    for _ in range(2):
        step(st)
    shapes = {}
    for a, z, c in itertools.product((0, 1), (0, 1), (0, 1)):
        job = _job(mlv, name, p, start, coeff, "f64")
        b = mlv.fused.Batch([job])
        if z and not b.plan["z_pass_split_available"]:
            b.close()
            continue
        b.set_plan(a, z, c)
        b.step(2)
        got = job.state()
        b.close()
        for f, g in zip(FIELDS[name], got):
            assert rel(g, st[f]) <= 1e-12, (a, z, c, f)
        for g, w in zip(got, shapes.setdefault(z, got)):
            np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("name", ["ddc", "mhd"])
def test_batch_over_both_z_passes(mlv, name):
    """One batch on both sides of the register pass's limit: each job's bits
    are its own run's."""
    def jobs():
        out = []
        for nx, nz in ((16, 512), (16, 1024), (32, 32), (64, 512)):
            p, start, coeff, _ = _problem(name, nx, nz, 4)
            out.append(_job(mlv, name, p, start, coeff, "f64"))
        return out

    together, alone = jobs(), jobs()
    b = mlv.fused.Batch(together)
    b.step(2)
    for j in alone:
        one = mlv.fused.Batch([j])
        one.step(2)
        one.close()
    for j, k in zip(together, alone):
        for g, w in zip(j.state(), k.state()):
            np.testing.assert_array_equal(g, w)
    b.close()
