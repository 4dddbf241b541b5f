"""The periodic finite check runs at the same steps however a run is cut into calls:
the first detection's step and count of a NaN forced from the host, a few steps after
the check was set, against a loop of simulator_calc()."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("every", [1, 3, 10, 64, 70, 150])
def test_step_of_the_check(precision, every):
    import mpifdtd_amd as m
    print(precision, every, flush=True)

    def run(parts):
        sim = m.Simulator(m.MPI_TM_UPML_2D, m.MIE_CYLINDER, m.field_info(60 * 20, 52 * 20, 20, 6, 500, 0, 400),
                          params=m.model_params(circle_radius_nm=200.0, circle_n=1.5), ntff_time=False,
                          precision=precision, T=4)
        try:
            sim.set_finite_check(every)
            sim.calc(5)
            for slot in (0, 2):
                a = sim.state(slot)
                a[30, 25] = np.nan
                sim.set_state(slot, a)
            for n in parts:
                sim.calc(n) if n else m.lib().simulator_calc()
            return sim.finite_status(), sim.check_finite(), sim.time
        finally:
            sim.set_finite_check(0)
            sim.finish()

    want = run([0] * 200)
    due = (5 // every + 1) * every  # the first check after the 5 steps; steps count from time 0
    assert want[0] is not None and want[0][0] == due - 1
    for parts in ([200], [1, 63, 64, 72], [9, 2, 189]):
        assert run(parts) == want, parts
