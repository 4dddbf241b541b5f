"""Simulator.fields() of a solver that another one of a different kind has followed:
its own fields, as its getters return them, and no array written at another's size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_fields_of_the_earlier_solver():
    import mpifdtd_amd as m
    L = m.lib()

    def make(solver, nx, ny):
        return m.Simulator(solver, m.MIE_CYLINDER, m.field_info(nx * 20, ny * 20, 20, 6, 500, 30, 40),
                           params=m.model_params(circle_radius_nm=200.0, circle_n=1.5), ntff_time=False)

    a = make(m.MPI_TM_UPML_2D, 60, 50)
    a.calc(40)
    first = a.fields()
    assert all(np.linalg.norm(f) > 0 for f in first)
    b = make(m.TE_UPML_2D, 41, 37)
    b.calc(11)
    for q in range(3):
        assert np.array_equal(a.fields()[q], first[q])
    assert [f.shape for f in b.fields()] == [(41, 37)] * 3
    assert np.array_equal(b.fields()[0], b.state(0))
    b.finish()
    with pytest.raises(RuntimeError):
        b.fields()
    assert np.array_equal(a.fields()[2], first[2])
    # a second solver of the same kind takes the first one's place
    c = make(m.MPI_TM_UPML_2D, 44, 40)
    with pytest.raises(RuntimeError):
        a.fields()
    c.finish()
