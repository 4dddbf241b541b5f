"""The FP64 blocked steps' second state, made by the first launch, in memory that held
something else: after a solver of the same size full of NaN, a new one's nine arrays,
edge ring and auxiliaries included, have the bits of the same run in fresh memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", range(8))
@pytest.mark.parametrize("nx,ny", [(45, 38), (150, 131)])
def test_second_state_in_used_memory(solver, nx, ny):
    import mpifdtd_amd as m
    print(solver, nx, ny, flush=True)

    def sim():
        return m.Simulator(solver, m.MIE_CYLINDER, m.field_info(nx * 20, ny * 20, 20, 6, 500, 30, 100),
                           params=m.model_params(circle_radius_nm=200.0, circle_n=1.5), ntff_time=False)

    def run():
        s = sim()
        try:
            for n in (8, 16, 9):
                s.calc(n)
            return [s.state(q) for q in range(9)]
        finally:
            s.finish()

    m.lib().fdtd_hip_trim()
    want = run()
    s = sim()
    bad = np.full((s.NPXa, s.NPYa), complex(np.nan, np.nan))
    try:
        s.calc(16)
        for q in range(9):
            s.set_state(q, bad)
        s.calc(16)  # (step by step)
        assert np.isnan(s.state(0)).any()
    finally:
        s.finish()
    # both states' blocks full of NaN: hand the first to the next solver's second state
    for _ in range(2):
        got = run()
        for a, b in zip(got, want):
            assert np.isfinite(a).all() and np.array_equal(a, b)
