"""Flux tile shapes where tile kernels run: under lbm_set_strips(0), and for
instances that need the reference's physical addressing (thin solids). All
shapes give bitwise identical states, those of the strips too where the
stencils have the same precision; with thin solids, whose tiles are evaluated
cell by cell in FP64, states within the bars of the two precisions. The
autotuner times shapes only where a tile kernel runs, and leaves shape and
default alone where none does."""
import numpy as np
import pytest

from uq_amd import cases
from uq_amd.lbm import rel_l2

pytestmark = pytest.mark.gpu


def _mirrored():
    c = cases.flat_plate(70, 36, plate_start=10, steps=8)
    c.params["mirror_north"] = 1
    c.params["mirror_east"] = 1
    return c


DECKS = {
    "couette": lambda: cases.couette(37, nx=45, u_wall=0.15, steps=8),
    "plate": lambda: cases.flat_plate(80, 40, plate_start=20, steps=8),
    "plate_mirrored": _mirrored,
    "riemann": lambda: cases.riemann(64, steps=8),
    "shear_rk1": lambda: cases.shear_wave(32, rk_method=0, steps=8),
}


BAR = {"fp64": 1e-12, "mixed": 1e-6}


def _states(lbm, case, prec, mode):
    out = []
    lbm.set_strips(mode)
    try:
        for shape in range(lbm.FLUX_SHAPES):
            lbm.set_flux_shape(prec, shape)
            s = lbm.Solver(case, prec)
            try:
                assert s.step(case.nsteps) == 0
                out.append(s.get_dist())
            finally:
                s.close()
    finally:
        lbm.set_flux_shape(prec, 0)
        lbm.set_strips(1)
    return out


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("name", list(DECKS))
def test_tile_shapes_equal(gpu_lib, name, prec):
    case = DECKS[name]()
    print(f"[tile shapes] {name} {prec}", flush=True)
    states = _states(gpu_lib, case, prec, 0)
    if prec == "fp64":
        states.append(_states(gpu_lib, case, prec, 1)[0])
    for k, (f, h) in enumerate(states):
        assert np.array_equal(f, states[0][0]) and np.array_equal(h, states[0][1]), k


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_thin_solid_takes_tiles_by_default(gpu_lib, prec):
    case = cases.obstacle(48, u0=0.1, block=(18, 20, 1, 8), steps=8)
    print(f"[tile shapes] thin solid {prec}", flush=True)
    states = _states(gpu_lib, case, prec, 1)
    for k, (f, h) in enumerate(states):
        assert max(rel_l2(f, states[0][0]), rel_l2(h, states[0][1])) <= BAR[prec], k


def _batch(lbm, prec, thin):
    members = [cases.couette(64, steps=9), cases.shear_wave(48, u0=0.1, steps=9)]
    if thin:
        members.append(cases.obstacle(48, u0=0.1, block=(18, 20, 1, 8), steps=9))
    solvers = [lbm.Solver(c, prec) for c in members]
    return solvers, lbm.Batch(solvers)


def _close(solvers, batch):
    batch.close()
    for s in solvers:
        s.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_autotune_without_tiles_keeps_the_shape(gpu_lib, prec):
    print(f"[tile shapes] autotune on strips {prec}", flush=True)
    gpu_lib.set_flux_shape(prec, 3)
    try:
        sa, ba = _batch(gpu_lib, prec, False)
        assert ba.step(2) == 0
        before = [s.get_dist() for s in sa]
        shape, ms = ba.autotune(steps=2)
        assert shape == 3 and len(set(ms)) == 1 and ms[0] > 0
        for s, (f, h) in zip(sa, before):
            f1, h1 = s.get_dist()
            assert np.array_equal(f, f1) and np.array_equal(h, h1) and s.info()["step"] == 2
        _close(sa, ba)
        sb, bb = _batch(gpu_lib, prec, False)  # the default is as it was
        assert bb.autotune(steps=1)[0] == 3
        _close(sb, bb)
    finally:
        gpu_lib.set_flux_shape(prec, 0)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("mode,thin", [(0, False), (1, True)])
def test_autotune_with_tiles(gpu_lib, prec, mode, thin):
    print(f"[tile shapes] autotune {prec} strips {mode} thin {thin}", flush=True)
    gpu_lib.set_strips(mode)
    try:
        sa, ba = _batch(gpu_lib, prec, thin)
        sb, bb = _batch(gpu_lib, prec, thin)
        assert ba.step(2) == 0 and bb.step(2) == 0
        shape, ms = ba.autotune(steps=2)
        assert len(set(ms)) > 1
        assert shape == min(k for k in range(gpu_lib.FLUX_SHAPES) if ms[k] <= min(ms) * 1.005)
        assert ba.step(7) == 0 and bb.step(7) == 0
        for k, (s, t) in enumerate(zip(sa, sb)):
            for x, y in zip(s.get_dist(), t.get_dist()):
                assert np.array_equal(x, y) if k < 2 else rel_l2(x, y) <= BAR[prec]
        _close(sa, ba)
        _close(sb, bb)
    finally:
        gpu_lib.set_strips(1)
        gpu_lib.set_flux_shape(prec, 0)
