"""The FP64 UPML solvers' blocked steps (several per launch) against the CPU
oracle: strips at the grid's edges, odd and non-square sizes, grids without any
interior strip, step counts that leave a partial block, one step per call, and
the changes that make a grid go on step by step.  All nine state arrays and the
NTFF accumulators at 1e-10 relative L2, the tolerance of the FP64 path.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-10
SOLVERS = {"tm": 2, "te": 3, "mpi_tm": 4, "mpi_te": 5}
H, PML, LAM, ANG = 20, 6, 500, 30
MIE = dict(circle_radius_nm=200.0, circle_n=1.5)


def _pair(solver, nx, ny, steps, **kw):
    import mpifdtd_amd as m
    from oracle import pyoracle as po
    print(f"{solver} {nx}x{ny} {steps} steps {kw}", flush=True)
    sim = m.Simulator(SOLVERS[solver], m.MIE_CYLINDER, m.field_info(nx * H, ny * H, H, PML, LAM, ANG, steps),
                      params=m.model_params(**MIE), **kw)
    ref = po.Sim(width_nm=nx * H, height_nm=ny * H, h_u_nm=H, pml=PML, lambda_nm=LAM, angle_deg=ANG, stepNum=steps,
                 solver=SOLVERS[solver], model=po.MIE_CYLINDER, **MIE)
    return sim, ref


def _same(sim, ref, slots=range(9)):
    for q in slots:
        assert rel_l2(sim.state(q), ref.field(q)) <= TOL, (q, rel_l2(sim.state(q), ref.field(q)))


@pytest.mark.parametrize("solver", sorted(SOLVERS))
@pytest.mark.parametrize("nx,ny,steps", [(41, 37, 83), (63, 97, 640), (140, 119, 641), (45, 301, 639)])
def test_blocks_against_oracle(solver, nx, ny, steps):
    sim, ref = _pair(solver, nx, ny, steps)
    try:
        sim.calc(steps)
        ref.step(steps)
        _same(sim, ref)
        if nx == 140:  # nearly square, as the oracle's NTFF needs
            for q in range(3):
                assert rel_l2(sim.ntff_time(q), ref.ntff_time(q)) <= TOL
    finally:
        sim.finish()


@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_calls_of_any_length_give_the_same_state(solver):
    sim, ref = _pair(solver, 140, 119, 640)
    try:
        for n in (1, 2, 7, 8, 9, 1, 64, 65, 483):
            sim.calc(n)
        ref.step(640)
        _same(sim, ref)
    finally:
        sim.finish()


@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_a_changed_state_goes_on_from_all_nine_arrays(solver):
    sim, ref = _pair(solver, 140, 119, 660)
    try:
        sim.calc(613)
        ref.step(613)
        for q in (0, 2):  # the field and its displacement are independent inputs of the next step
            a = 0.5 * sim.state(q)
            sim.set_state(q, a)
            ref.set_field(q, a)
        sim.calc(47)
        ref.step(47)
        _same(sim, ref)
        sim.reset()
        ref.reset()
        sim.calc(600)
        ref.step(600)
        _same(sim, ref)
    finally:
        sim.finish()


def test_point_source_in_a_frame_strip():
    """The source cell of a small grid lies in a strip that runs the full recurrences."""
    import mpifdtd_amd as m
    from oracle import pyoracle as po
    args = (31 * H, 30 * H, H, PML, LAM, 0, 90)
    sim = m.Simulator(m.MPI_TM_UPML_2D, m.NO_MODEL, m.field_info(*args), point_source=True, ntff_time=False)
    ref = po.Sim(width_nm=args[0], height_nm=args[1], h_u_nm=H, pml=PML, lambda_nm=LAM, angle_deg=0, stepNum=90,
                 solver=4, model=po.NO_MODEL, point_source=1)
    try:
        sim.calc(90)
        ref.step(90)
        _same(sim, ref)
    finally:
        sim.finish()
