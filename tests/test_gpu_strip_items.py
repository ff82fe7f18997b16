"""Work items of the strip flux kernels: one wavefront per item and direction,
the rows per item (1 to 32) chosen by the size of the launch group. The item
edges (rows per item, the last partial strip and item, items of one row next
to a solid, grids of fewer items than XCDs) must not show: strips (the
default) equal the tile kernels bit for bit, and a member of a large batch,
whose items are longer, equals its lone run. (Items of up to 32 rows:
tests/test_gpu_long_items.py.)"""
import numpy as np
import pytest

from uq_amd import cases

pytestmark = pytest.mark.gpu


def _deck(kind, nx, ny, flux, rk):
    if kind == "couette":
        return cases.couette(ny, nx=nx, u_wall=0.12, flux_method=flux, rk_method=rk, steps=6)
    if kind == "plate":
        c = cases.flat_plate(nx, ny, plate_start=nx // 3, flux_method=flux, rk_method=rk, steps=6)
        c.params["mirror_east"] = 1
        return c
    c = cases.riemann(max(nx, ny), steps=6, flux_method=flux, rk_method=rk, cfl=0.1)
    c.bnd = np.ascontiguousarray(c.bnd[:nx, :ny])
    return c


def _run(lbm, case, prec, mode):
    lbm.set_strips(mode)
    try:
        s = lbm.Solver(case, prec)
        try:
            assert s.step(6) == 0
            return s.get_dist()
        finally:
            s.close()
    finally:
        lbm.set_strips(1)


# sides: below, at and beyond one strip (58 columns), one item (one row at
# the smallest), the window (7 rows) and the 64 lanes; rows not a multiple of any item
SIDES = [(5, 6), (58, 9), (59, 33), (64, 64), (117, 65), (175, 130)]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,flux,rk", [("couette", 1, 1), ("couette", 0, 0), ("plate", 0, 1), ("riemann", 1, 1),
                                          ("riemann", 0, 3)])
def test_items_equal_tiles(gpu_lib, kind, flux, rk, prec):
    for nx, ny in SIDES:
        if kind == "plate" and nx < 16:
            continue
        case = _deck(kind, nx, ny, flux, rk)
        print(f"[strip items] {kind} {nx}x{ny} flux {flux} rk {rk} {prec}", flush=True)
        fs, hs = _run(gpu_lib, case, prec, 1)
        ft, ht = _run(gpu_lib, case, prec, 0)
        assert np.array_equal(fs, ft) and np.array_equal(hs, ht), (nx, ny)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_member_of_a_large_batch_equals_alone(gpu_lib, prec):
    """The batch's items have some ten rows, the lone solver's one or two."""
    small = [cases.couette(41, nx=61, steps=8), cases.shear_wave(66, u0=0.1, steps=8)]
    alone = []
    for c in small:
        s = gpu_lib.Solver(c, prec)
        assert s.step(8) == 0
        alone.append(s.get_dist())
        s.close()
    solvers = [gpu_lib.Solver(c, prec) for c in small + [cases.shear_wave(700, u0=0.1, steps=8)]]
    b = gpu_lib.Batch(solvers)
    try:
        assert b.step(8) == 0
        for s, (fa, ha) in zip(solvers, alone):
            f, h = s.get_dist()
            assert np.array_equal(f, fa) and np.array_equal(h, ha)
    finally:
        b.close()
        for s in solvers:
            s.close()
