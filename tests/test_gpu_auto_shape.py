"""The launch shape that FAST_LAUNCH_AUTO picks for FP32 grids (1 merged, 2 split, 8
split with 16-wavefront UPML tiles, 9 those on two streams), on either side of its
lines where the two shapes' times are over 10 % apart, and its fields against the
merged launch's, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # solver (2 TM, 3 TE, 4 MPI TM, 5 MPI TE), cells, T, R, running DFT, shape
    (3, 80, 80, 1, 16, False, 1), (3, 80, 80, 4, 16, False, 1), (3, 80, 80, 8, 16, False, 1), (3, 300, 260, 8, 16, False, 9),
    (3, 500, 400, 4, 16, False, 1), (3, 200, 200, 8, 8, False, 1), (3, 1056, 1056, 8, 16, False, 8),
    (3, 1400, 1200, 1, 16, False, 1), (3, 1056, 1056, 2, 4, False, 2), (3, 1040, 960, 4, 16, True, 9),
    (2, 1056, 1056, 4, 16, False, 1), (2, 1056, 1056, 8, 16, True, 8), (2, 2640, 2560, 8, 16, False, 1),
    (4, 1056, 1056, 8, 16, False, 1), (4, 1400, 1200, 8, 16, True, 8), (4, 3000, 2400, 8, 16, False, 1),
    (5, 1056, 1056, 1, 16, False, 1), (5, 1056, 1056, 8, 16, False, 8), (5, 2000, 1500, 4, 16, False, 2),
    (5, 400, 300, 8, 16, False, 1),
]


@pytest.mark.parametrize("solver,nx,ny,T,R,dft,shape", CASES)
def test_shape(solver, nx, ny, T, R, dft, shape):
    import mpifdtd_amd as m
    print(solver, nx, ny, T, R, dft, flush=True)
    fields = []
    for mode in (0, 1):
        sim = m.Simulator(solver, m.MIE_CYLINDER, m.field_info(nx * 5, ny * 5, 5, 10, 500, 0, 100),
                          params=m.model_params(circle_radius_nm=0.14 * min(nx, ny) * 5, circle_n=1.6), ntff_time=False,
                          precision="fp32", T=T, R=R)
        try:
            sim.set_launch_mode(mode)
            if dft:
                sim.set_dft([500.0])
            sim.calc(2 * T)
            fields.append(sim.state(0 if solver % 2 == 0 else 3))
            assert sim.launch_mode() == (mode or shape)
        finally:
            sim.finish()
    assert np.array_equal(*fields)
