"""FP64 grids with cells whose 1/eps is zero (perfect conductors) or so small that the
displacement cannot be formed from the field: the nine arrays against a NumPy
restatement, with calls of one step and of many, and again after a reset and after a
map of ordinary values.  1e-10 of each array's norm, the tolerance of the FP64 path."""
import numpy as np
import pytest

import gridapi as ga
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ga.TM, ga.TE])
@pytest.mark.parametrize("flavour", [ga.MPI, ga.PLAIN])
@pytest.mark.parametrize("big", [np.inf, 1e9])
def test_large_permittivity(mode, flavour, big):
    nx, ny, n = 45, 38, 19
    print(f"mode {mode} flavour {flavour} eps {big}", flush=True)
    g = ga.Grid(mode, flavour, nx, ny)
    try:
        eps = np.ones((3,) + g.shape)
        eps[:, 12:20, 9:16] = 2.25
        eps[:, 17:23, 14:22] = big
        eps[:, 0, 0] = np.inf  # a cell that is never updated
        t0 = 5 if flavour == ga.MPI else 470  # near the pulse's peak
        p = g.params(t0, n)
        for e, reset in ((eps, False), (eps, True), (np.minimum(eps, 4.0), True)):
            if reset:
                g.reset()
            g.set_eps(e)
            g.steps(p)
            want = ga.reference(mode, flavour, nx, ny, e, p)
            assert np.linalg.norm(want[0 if mode == ga.TM else 3]) > 0.1
            for q in range(9):
                assert rel_l2(g.field(q), want[q]) <= 1e-10, (q, rel_l2(g.field(q), want[q]))
        # set while steps are taken, the wave's next steps one by one
        g.set_eps(eps)
        before = [g.field(q) for q in range(9)]
        assert all(np.isfinite(f).all() for f in before)
        for q in g.params(t0 + n, 3):
            g.step(q)
        got = g.field(0 if mode == ga.TM else 3)
        assert np.isfinite(got).all()
    finally:
        g.close()
