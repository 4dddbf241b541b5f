"""The NTFF binning records that the device sorts: every contour sample lands in the
time-domain accumulators exactly once and on its bins.  The running DFT of the
contour, which uses no records, has to equal the DFT of the accumulators, to 1e-10
relative L2 (both FP64 on the same samples), with every contour cell excited by a
random state (set after as many dark steps as the longest shift, and that many before the
end, so that no bin leaves its row).  Sizes: a small contour; one whose offsets leave gaps between the sides
longer than a part may span; a long one sorted in more than one pass.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [2, 3, 4, 5])
@pytest.mark.parametrize("nx,ny", [(46, 49), (1100, 60), (60, 7001)])
def test_every_sample_is_binned_once(solver, nx, ny):
    import mpifdtd_amd as m
    print(solver, nx, ny, flush=True)
    h, pml, steps, T = 10, 6, 11, 8
    dark = 8 * (int(np.hypot(nx, ny) / 0.7071) // 8 + 1)
    sim = m.Simulator(solver, m.NO_MODEL, m.field_info(nx * h, ny * h, h, pml, 500, 0, steps + 2 * dark),
                      precision="fp32", T=T)
    try:
        sim.calc(dark)
        rng = np.random.default_rng(nx + solver)
        for q in (0, 3, 6):
            a = rng.standard_normal((sim.NPXa, sim.NPYa)) + 1j * rng.standard_normal((sim.NPXa, sim.NPYa))
            if sim.off:
                a[[0, -1], :] = 0
                a[:, [0, -1]] = 0
            sim.set_state(q, a)
        lam = np.array([433.0, 700.0])
        sim.set_dft(lam)
        sim.calc(steps)
        got = sim.dft()
        w = 0.7071 * 2 * np.pi / (lam / h)
        e = np.exp(1j * np.outer(w, np.arange(sim.arraySize)))
        for q in range(3):
            U = sim.ntff_time(q)
            assert rel_l2(e @ U.T, got[:, q]) <= 1e-10, (q, rel_l2(e @ U.T, got[:, q]))
    finally:
        sim.finish()
