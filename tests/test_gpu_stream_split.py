"""The FP64 split-field and non-standard solvers' blocked steps against the CPU
oracle: every kept array, odd and non-square grids, partial blocks, calls of any
length, and a changed state, at 1e-10 relative L2 (the tolerance of the FP64 path).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-10
SOLVERS = {"split_tm": 0, "split_te": 1, "ns_tm": 6, "ns_te": 7}
SLOTS = {"split_tm": (0, 1, 2, 3, 6), "split_te": (0, 3, 6, 7, 8), "ns_tm": (0, 1, 2, 3, 6), "ns_te": (0, 3, 6, 7, 8)}
H, PML, LAM, ANG = 20, 6, 500, 30
MIE = dict(circle_radius_nm=200.0, circle_n=1.5)


def _pair(solver, nx, ny, steps):
    import mpifdtd_amd as m
    from oracle import pyoracle as po
    print(f"{solver} {nx}x{ny} {steps} steps", flush=True)
    sim = m.Simulator(SOLVERS[solver], m.MIE_CYLINDER, m.field_info(nx * H, ny * H, H, PML, LAM, ANG, steps),
                      params=m.model_params(**MIE))
    ref = po.Sim(width_nm=nx * H, height_nm=ny * H, h_u_nm=H, pml=PML, lambda_nm=LAM, angle_deg=ANG, stepNum=steps,
                 solver=SOLVERS[solver], model=po.MIE_CYLINDER, **MIE)
    return sim, ref


def _same(solver, sim, ref):
    for q in SLOTS[solver]:
        assert rel_l2(sim.state(q), ref.field(q)) <= TOL, (q, rel_l2(sim.state(q), ref.field(q)))


@pytest.mark.parametrize("solver", sorted(SOLVERS))
@pytest.mark.parametrize("nx,ny,steps", [(41, 37, 83), (63, 97, 200), (140, 119, 201), (45, 301, 199)])
def test_blocks_against_oracle(solver, nx, ny, steps):
    sim, ref = _pair(solver, nx, ny, steps)
    try:
        sim.calc(steps)
        ref.step(steps)
        _same(solver, sim, ref)
    finally:
        sim.finish()


@pytest.mark.parametrize("solver", sorted(SOLVERS))
def test_calls_of_any_length_and_a_changed_state(solver):
    sim, ref = _pair(solver, 140, 119, 200)
    try:
        for n in (1, 2, 3, 4, 5, 7, 8, 9, 64, 37):
            sim.calc(n)
            ref.step(n)
        _same(solver, sim, ref)
        for q in SLOTS[solver][:2]:
            a = 0.5 * sim.state(q)
            sim.set_state(q, a)
            ref.set_field(q, a)
        sim.calc(13)
        ref.step(13)
        _same(solver, sim, ref)
        sim.reset()
        ref.reset()
        sim.calc(100)
        ref.step(100)
        _same(solver, sim, ref)
    finally:
        sim.finish()
