"""Strip items of 2 to 32 rows: the rows per item follow from the size of the
launch group, so small decks are stepped in a batch beside one large uniform
instance, whose size brings the items to the wanted length. Every small member
must equal its lone run on the tile kernels bit for bit (mixed precision far
from the reference equilibrium, plate and shock deck, whose strip stencils are
FP64 in a large group and whose tile stencils FP32: the lone run on short items
with FP64 stencils): the row table and the
windows of long items, their last partial item, rows next to solids, mirrored
and periodic edges, for the fused FP64 step, the FP64 strip fluxes of the
one-stage stepper and the two FP32 strip kernels."""
import numpy as np
import pytest

from uq_amd import cases

pytestmark = pytest.mark.gpu

STEPS = 6


def _members(rk):
    plate = cases.flat_plate(117, 65, plate_start=40, flux_method=0, rk_method=rk, steps=STEPS)
    plate.params["mirror_north"] = 1
    shock = cases.riemann(130, steps=STEPS, rk_method=rk, cfl=0.1)
    shock.bnd = np.ascontiguousarray(shock.bnd[:60])
    return [cases.couette(33, nx=61, rk_method=rk, steps=STEPS), plate,
            cases.obstacle(65, block=(30, 20, 9, 12), u0=0.05, rk_method=rk, steps=STEPS),
            cases.shear_wave(130, u0=0.1, rk_method=rk, steps=STEPS), shock]


def _large(nx, ny, rk):
    c = cases.riemann(16, steps=STEPS, rk_method=rk)
    c.bnd = np.full((nx, ny), c.bnd[0, 0], dtype=c.bnd.dtype)
    return c


# sides of the large instance; the rule gives a batch of all members beside it items
# of 8, 8, 30 and 32 rows for the strip fluxes, 2, 7, 31 and 32 for the fused step
# and the FP32 flux with moment sums
@pytest.mark.parametrize("nx,ny", [(464, 176), (58, 2000), (116, 46500), (116, 68500)])
@pytest.mark.parametrize("prec,rk", [("fp64", 1), ("fp64", 0), ("mixed", 1)])
def test_members_equal_tiles(gpu_lib, prec, rk, nx, ny):
    lbm = gpu_lib
    members = _members(rk)
    far = [prec == "mixed" and c.name.startswith(("plate", "riemann")) for c in members]
    print(f"[long items] {prec} rk {rk} beside {nx}x{ny}", flush=True)
    alone = []
    try:
        for c, f64 in zip(members, far):
            lbm.set_strips(2 if f64 else 0)
            s = lbm.Solver(c, prec)
            assert s.step(STEPS) == 0
            alone.append(s.get_dist())
            s.close()
    finally:
        lbm.set_strips(1)
    solvers = [lbm.Solver(c, prec) for c in members + [_large(nx, ny, rk)]]
    batch = lbm.Batch(solvers)
    lbm.set_strips(2 if prec == "mixed" else 1)
    try:
        assert batch.step(STEPS) == 0
        for c, s, (fa, ha) in zip(members, solvers, alone):
            f, h = s.get_dist()
            assert np.array_equal(f, fa) and np.array_equal(h, ha), c.name
    finally:
        lbm.set_strips(1)
        batch.close()
        for s in solvers:
            s.close()
