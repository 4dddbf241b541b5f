"""The far field of the running DFT by the launches for short contours, few frequencies
and the rest: one frequency by itself and among five, on grids whose contours are a few
cells below and above the lines.  The sums differ in order alone: 1e-11 of the norm.
(test_gpu_dft.py compares the DFT with the per-step NTFF's accumulators.)"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [2, 3, 4, 5])
@pytest.mark.parametrize("nx,ny", [(60, 47), (217, 205), (222, 208), (300, 281)])
def test_launches_agree(solver, nx, ny):
    import mpifdtd_amd as m
    print(solver, nx, ny, flush=True)
    lams = [450.0, 480.0, 500.0, 550.0, 620.0]

    def run(l):
        sim = m.Simulator(solver, m.MIE_CYLINDER, m.field_info(nx * 20, ny * 20, 20, 8, 500, 30, 620),
                          params=m.model_params(circle_radius_nm=0.2 * min(nx, ny) * 20, circle_n=1.5), ntff_time=False)
        try:
            sim.set_dft(l)
            sim.calc(620)
            return sim.dft()
        finally:
            sim.finish()

    assert rel_l2(run([500.0])[0], run(lams)[2]) <= 1e-11
