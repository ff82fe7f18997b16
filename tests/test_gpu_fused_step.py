"""The RK3 step of FP64 storage in two launches (the state kept only in the
stage values between the steps of a sequence) against the tile kernels (four
launches, the state in memory after every step), bit for bit: however a run is
cut into sequences (the first, the last two and the graph-replayed steps are
launched differently), for sides below, at and beyond a strip, for periodic,
mirrored and open edges, walls, stretched spacings and a temperature-dependent
viscosity, and for a member that fails inside a sequence."""
import numpy as np
import pytest

from uq_amd import cases

pytestmark = pytest.mark.gpu


def _deck(kind):
    if kind == "couette":
        return cases.stretched(cases.couette(61, nx=59, u_wall=0.12), amp=0.3)
    if kind == "plate":
        c = cases.flat_plate(130, 49, plate_start=40, flux_method=0)
        c.params["mirror_east"] = 1
        return c
    if kind == "block":
        c = cases.obstacle(75, block=(25, 31, 9, 7), u0=0.05)
        T = float(c.props["temp"][0])
        c.meta["viscosity"] = dict(model="vhs", mu_ref=c.params["mu"], T_ref=T, param=0.2)
        return c
    if kind == "small":
        return cases.shear_wave(7, u0=0.1)
    return cases.riemann(97, cfl=0.1)


def _run(lbm, case, cuts, mode=1, graphs=True):
    lbm.set_strips(mode)
    lbm.set_graphs(graphs)
    try:
        s = lbm.Solver(case, "fp64")
        try:
            for n in cuts:
                assert s.step(n) == 0
            return s.get_dist()
        finally:
            s.close()
    finally:
        lbm.set_strips(1)
        lbm.set_graphs(True)


@pytest.mark.parametrize("kind", ["couette", "plate", "block", "small", "riemann"])
def test_sequences_equal_tiles(gpu_lib, kind):
    case, total = _deck(kind), 22
    ft, ht = _run(gpu_lib, case, [total], mode=0)
    # one and two steps alone, graphs of eight steps with 0, 1 or more steps around them
    for cuts in ([22], [1, 2, 19], [10, 11, 1], [9, 3, 10], [1] * 4 + [18]):
        print(f"[fused] {kind} {cuts}", flush=True)
        f, h = _run(gpu_lib, case, cuts)
        assert np.array_equal(f, ft) and np.array_equal(h, ht), cuts
    f, h = _run(gpu_lib, case, [22], graphs=False)
    assert np.array_equal(f, ft) and np.array_equal(h, ht)


@pytest.mark.parametrize("n", [1, 2, 3, 12])
def test_residual_of_a_sequence(gpu_lib, n):
    """The residual compares the states of the last two steps."""
    case, res = cases.couette(61, nx=59, u_wall=0.12), []
    for mode in (0, 1):
        gpu_lib.set_strips(mode)
        try:
            s = gpu_lib.Solver(case, "fp64")
            try:
                s.step(3)
                res.append(s.step(n, want_residual=True))
            finally:
                s.close()
        finally:
            gpu_lib.set_strips(1)
    assert res[0] == res[1] and res[0][0] == 0


@pytest.mark.parametrize("ratio,cfl", [(400.0, 0.1), (5.0, 0.1), (3.0, 0.5)])
def test_failing_member_of_a_batch(gpu_lib, ratio, cfl):
    """A member that fails inside a sequence (at step 2, 15 or 22) keeps the
    state of the failing step, the others run on."""
    bad = cases.riemann(80, cfl=cfl)
    bad.props["pressure"] = bad.props["pressure"] * np.array([ratio, 1.0, 1.0, 1.0])
    bad.props["temp"] = bad.props["pressure"] / (bad.props["density"] * bad.params["R"])
    got = []
    for mode in (0, 1):
        gpu_lib.set_strips(mode)
        try:
            solvers = [gpu_lib.Solver(c, "fp64") for c in (bad, cases.shear_wave(66, u0=0.1))]
            b = gpu_lib.Batch(solvers)
            try:
                status = b.step(60)
                got.append((status, [s.info()["step"] for s in solvers], [s.get_dist() for s in solvers]))
            finally:
                b.close()
                for s in solvers:
                    s.close()
        finally:
            gpu_lib.set_strips(1)
    assert got[0][:2] == got[1][:2]
    assert got[0][0] == 1 and 0 < got[0][1][0] < 60 and got[0][1][1] == 60
    for (fa, ha), (fb, hb) in zip(got[0][2], got[1][2]):
        assert np.array_equal(fa, fb, equal_nan=True) and np.array_equal(ha, hb, equal_nan=True)
