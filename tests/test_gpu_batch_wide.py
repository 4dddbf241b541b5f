"""Batches with 48-row UPML tiles against those with 32-row tiles, bit for bit, and
contour samples handed on for several blocks at once against other cuts of the run.

The tiles differ in which workgroup computes a cell, not in its arithmetic.  The
samples are summed into FP64 accumulators in another order (FP32 solvers: the same
samples, 1e-12); FP64 solvers' blocks follow the calls, so theirs agree to the FP64
path's 1e-10.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

# solver, nx, ny, pml, steps: no interior tile, one tile and a bit, odd and non-square, wide
GRIDS = [(4, 44, 60, 10, 63), (5, 131, 97, 10, 71), (4, 67, 203, 16, 80), (5, 260, 75, 6, 47)]


@pytest.mark.parametrize("grids", [GRIDS, GRIDS[:1], GRIDS[1::2]], ids=["both", "one_tm", "te"])
@pytest.mark.parametrize("T,R", [(1, 4), (8, 8), (10, 16), (15, 16)])
def test_wide_upml_tiles(T, R, grids):
    import mpifdtd_amd as m
    from mpifdtd_amd import batch as B
    print(f"T {T} R {R} {len(grids)} instances", flush=True)
    items = [B.item(s, m.MIE_CYLINDER, nx * 20, ny * 20, 20, pml, 500, 30, st, circle_radius_nm=200.0, circle_n=1.5)
             for (s, nx, ny, pml, st) in grids]

    def run(shapes):
        with B.Batch(items, T=T, R=R) as b:
            for shape in shapes:
                b.set_launch_mode(shape)
                b.run_blocks(2)
                b.sync()
            b.run()
            return [b.field(i, q) for i in range(len(grids)) for q in range(9)]

    narrow = run([2])
    for shapes in ([5], [6], [5, 3, 4, 2, 7]):
        for a, c in zip(narrow, run(shapes)):
            assert np.array_equal(a, c), shapes


@pytest.mark.parametrize("solver,prec,T", [(4, "fp64", None), (3, "fp64", None), (5, "fp32", 3), (2, "fp32", 8), (4, "fp32", 15)])
def test_samples_of_several_blocks(solver, prec, T):
    import mpifdtd_amd as m
    print(f"solver {solver} {prec} T {T}", flush=True)

    def run(parts):
        sim = m.Simulator(solver, m.MIE_CYLINDER, m.field_info(120 * 20, 110 * 20, 20, 8, 500, 30, 400),
                          params=m.model_params(circle_radius_nm=200.0, circle_n=1.5), precision=prec,
                          **({} if T is None else dict(T=T, R=16)))
        try:
            for n in parts:
                sim.calc(n)
            return [sim.ntff_time(q) for q in range(3)]
        finally:
            sim.finish()

    whole = run([400])
    for parts in ([1, 8, 9, 17, 40, 325], [16, 15, 64, 65, 240]):
        for a, c in zip(whole, run(parts)):
            assert np.linalg.norm(a) == 0 if not np.any(c) else rel_l2(c, a) <= (1e-10 if prec == "fp64" else 1e-12)
