"""The residual of a step call in which the solver fails (reference runOne,
cpuLBM.cpp:2322-2331: the RMS change of T over the last step taken). The tile
kernels have the state of every step in memory; the FP64 RK3 step in two
launches writes it in the last two steps of a sequence and at the failing one,
so a failure at an inner step has to be taken again up to the step before.
Status, residual, step count and state equal those of the tile kernels bit for
bit: failures at the first, an even and an odd step of the call, at its last
step, next to its last step and well inside it (with and without captured
graphs of steps before), on a new solver and behind other calls, through both
step entry points."""
import ctypes as C

import numpy as np
import pytest

from uq_amd import cases

pytestmark = pytest.mark.gpu


def _failing(ratio, cfl):
    c = cases.riemann(80, cfl=cfl)
    c.props["pressure"] = c.props["pressure"] * np.array([ratio, 1.0, 1.0, 1.0])
    c.props["temp"] = c.props["pressure"] / (c.props["density"] * c.params["R"])
    return c


def _step(lbm, s, n, entry):
    res = C.c_double(-1.0)
    f = getattr(lbm.lib(), entry)
    f.argtypes = [C.c_void_p, C.c_int32, C.c_int32, C.POINTER(C.c_double)]
    return f(s.handle, n, 1, C.byref(res)), res.value


def _run(lbm, case, mode, calls, entry):
    lbm.set_strips(mode)
    try:
        s = lbm.Solver(case, "fp64")
        try:
            got = [_step(lbm, s, n, entry) for n in calls]
            return got, s.info()["step"], s.get_dist()
        finally:
            s.close()
    finally:
        lbm.set_strips(1)


@pytest.mark.parametrize("entry", ["lbm_step", "lbm_step_noalloc"])
@pytest.mark.parametrize("ratio,cfl,at", [(400.0, 0.1, 2), (5.0, 0.1, 14), (3.0, 0.5, 22)])
def test_residual_of_a_failing_call_equals_tiles(gpu_lib, ratio, cfl, at, entry):
    case = _failing(ratio, cfl)
    assert _run(gpu_lib, case, 0, [60], entry)[1] == at
    # the failing step `at` as the last step of the call, next to the last, and inside it;
    # behind calls that leave it at an odd or even place, or first, in its own call
    for calls in ([at], [at + 1], [60], [1, 60], [at - 1, 9], [at - 1, 1], [1] * (at - 2) + [2]):
        print(f"[failing residual] step {at} calls {calls} {entry}", flush=True)
        want = _run(gpu_lib, case, 0, calls, entry)
        got = _run(gpu_lib, case, 1, calls, entry)
        assert want[0][-1][0] == 1 and want[1] == at
        assert got[0] == want[0] or np.array_equal(got[0], want[0], equal_nan=True), (calls, got[0][-1], want[0][-1])
        assert got[1] == at
        for a, b in zip(got[2], want[2]):
            assert np.array_equal(a, b, equal_nan=True)
    # a failed solver takes no further step
    s = gpu_lib.Solver(case, "fp64")
    try:
        assert _step(gpu_lib, s, 60, entry)[0] == 1 and _step(gpu_lib, s, 5, entry)[0] == 1
        assert s.info()["step"] == at
    finally:
        s.close()
