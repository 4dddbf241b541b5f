"""FP64 UPML blocked steps with a scatterer in every cell, at sizes whose strips end
inside, at and past the grid's edge, so that a strip's halo lanes and those past them
hold scatterers: the nine arrays against a NumPy restatement at 1e-10 of each array's
norm, the tolerance of the FP64 path."""
import numpy as np
import pytest

import gridapi as ga
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ga.TM, ga.TE])
@pytest.mark.parametrize("flavour", [ga.MPI, ga.PLAIN])
@pytest.mark.parametrize("nx,ny", [(24, 150), (70, 131), (33, 62), (50, 129)])
def test_random_permittivity(mode, flavour, nx, ny):
    print(f"mode {mode} flavour {flavour} {nx}x{ny}", flush=True)
    g = ga.Grid(mode, flavour, nx, ny)
    try:
        eps = 1.0 + 2.0 * np.random.default_rng(nx).random((3,) + g.shape)
        g.set_eps(eps)
        p = g.params(5 if flavour == ga.MPI else 470, 19)
        g.steps(p)
        want = ga.reference(mode, flavour, nx, ny, eps, p)
        for q in range(9):
            assert rel_l2(g.field(q), want[q]) <= 1e-10, (q, rel_l2(g.field(q), want[q]))
    finally:
        g.close()
