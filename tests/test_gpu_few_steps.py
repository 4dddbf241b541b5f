"""Calls of a few FP64 steps, which go by the kernels of a step, between runs that go
in blocks: on a small grid a loop of simulator_calc() gives the bits of those kernels
(a grid that set_state has sent to them), and runs cut in any way agree with it to
1e-10 of each array's norm, the tolerance of the FP64 path, with the per-step NTFF and
the running DFT beside them."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

KEPT = {0: (0, 1, 2, 3, 6), 1: (0, 3, 6, 7, 8), 6: (0, 1, 2, 3, 6), 7: (0, 3, 6, 7, 8)}  # split-field, NS
CUTS = ([8, 1, 9, 2, 16, 3, 1, 24, 5, 11], [1, 16, 1, 1, 23, 4, 6, 7, 21], [80])


def run(solver, parts, ntff, by_step=False, nx=70, ny=61, radius=200.0):
    """(arrays, NTFF accumulators, DFT) after calls of `parts` steps, 0: one simulator_calc()."""
    import mpifdtd_amd as m
    sim = m.Simulator(solver, m.MIE_CYLINDER, m.field_info(nx * 20, ny * 20, 20, 6, 500, 30, 100),
                      params=m.model_params(circle_radius_nm=radius, circle_n=1.5), ntff_time=bool(ntff & 1))
    try:
        if ntff & 2:
            sim.set_dft([450.0, 500.0, 620.0])
        if by_step:
            sim.set_state(0, sim.state(0))
        for n in parts:
            sim.calc(n) if n else m.lib().simulator_calc()
        arrays = [sim.state(q) for q in KEPT.get(solver, range(9))]
        return arrays, [sim.ntff_time(q) for q in range(3)] if ntff & 1 else [], [sim.dft()] if ntff & 2 else []
    finally:
        sim.finish()


@pytest.mark.parametrize("solver", range(8))
def test_a_loop_of_single_steps_has_the_bits_of_the_step_kernels(solver):
    print("solver", solver, flush=True)
    want = run(solver, [0] * 25, 0, by_step=True)[0]
    for parts in ([0] * 25, [1] * 25, [2] * 12 + [0]):
        for a, b in zip(run(solver, parts, 0)[0], want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("solver,ntff", [(s, n) for s in range(8) for n in ((0, 1, 2, 3) if 2 <= s <= 5 else (0, 2))])
def test_cuts_of_a_run(solver, ntff):
    print("solver", solver, "ntff", ntff, flush=True)
    want = run(solver, [0] * 80, ntff, by_step=True)
    for parts in CUTS:
        got = run(solver, parts, ntff)
        for g, w in zip(got, want):
            for a, b in zip(g, w):
                assert rel_l2(a, b) <= 1e-10, (parts, rel_l2(a, b))


@pytest.mark.parametrize("solver", (2, 3, 4, 5))
def test_cuts_with_a_scatterer_up_to_the_absorbing_layer(solver):
    want = run(solver, [0] * 80, 1, by_step=True, radius=640.0)
    for parts in CUTS:
        for g, w in zip(run(solver, parts, 1, radius=640.0), want):
            for a, b in zip(g, w):
                assert rel_l2(a, b) <= 1e-10, (parts, rel_l2(a, b))
