"""FP64 UPML blocked steps where the frame and interior strips run as two launches (more
than 512 strips: 16000 rows of 80 columns make over 600 of the longest), with a
scatterer in every cell, an absorbing layer on the rows and the running DFT's contour
samples, against the kernels of a step (a grid that set_field has sent to them): the
nine arrays and the DFT at 1e-10 relative L2, the tolerance of the FP64 path."""
import numpy as np
import pytest

import gridapi as ga
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ga.TM, ga.TE])
@pytest.mark.parametrize("flavour", [ga.MPI, ga.PLAIN])
def test_two_launches(mode, flavour):
    nx, ny, n = 16000, 80, 21
    print(f"mode {mode} flavour {flavour}", flush=True)
    eps = 1.0 + 2.0 * np.random.default_rng(1).random((nx + 2, ny + 2))

    def run(by_step):
        g = ga.Grid(mode, flavour, nx, ny, pml=10)
        try:
            x, y = g.shape
            g.set_eps([eps[:x, :y], eps[::-1, :][:x, :y], eps[:x, :y]])
            g.set_dft([0.2, 0.31])
            if by_step:
                g.set_field(0, np.zeros(g.shape))
            # almost along the columns: the pulse reaches every row
            g.steps(g.params(5 if flavour == ga.MPI else 470, n, angle=88.0))
            return [g.field(q) for q in range(9)] + [g.dft()]
        finally:
            g.close()

    want = run(True)
    got = run(False)
    for q in range(10):
        assert rel_l2(got[q], want[q]) <= 1e-10, (q, rel_l2(got[q], want[q]))
        rows = np.abs(want[q]).sum(axis=tuple(range(1, want[q].ndim)))
        if q < 9 and rows.size > 100:
            assert np.count_nonzero(rows) > 15000  # the comparison covers the grid
