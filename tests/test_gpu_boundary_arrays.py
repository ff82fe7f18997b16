"""The boundary's arrays ([x][y][i] distributions, [x][y] fields): transposed
on the device in 16 x 16 and 32 x 32 cell tiles and copied in 2 MiB pieces, so
grids below, at and beyond a tile and a piece. FP64: distributions put in come
back bit for bit. Mixed: every stored deviation is rounded to FP32 once and a
cell's rounding defects (13 of them at most) are moved to f0, f1..f4 and h0,
so a value is off by at most 14 roundings of the cell's largest deviation,
while the cell's conserved sums come back in FP64. Fields equal the moments of
the distributions that come back."""
import threading

import numpy as np
import pytest

from uq_amd import cases

pytestmark = pytest.mark.gpu

EX = np.array([0, 1, 0, -1, 0, 1, -1, -1, 1, 2, 0, -2, 0])
EY = np.array([0, 0, 1, 0, -1, 1, 1, -1, -1, 0, 2, 0, -2])
GRIDS = [(4, 5), (16, 16), (17, 33), (64, 31), (130, 70), (601, 250)]


def _case(nx, ny):
    return cases.couette(ny, nx=nx, steps=1)


def _values(f0, h0, seed):
    rng = np.random.default_rng(seed)
    return f0 * (1 + 0.1 * rng.uniform(-1, 1, f0.shape)), h0 * (1 + 0.1 * rng.uniform(-1, 1, h0.shape))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_round_trip_and_fields(gpu_lib, nx, ny, prec):
    s = gpu_lib.Solver(_case(nx, ny), prec)
    try:
        f0, h0 = s.get_dist()
        f, h = _values(f0, h0, nx)
        s.set_dist(f, h)
        fb, hb = s.get_dist()
        m = s.get_macro()
        c = s.info()["c"]
    finally:
        s.close()
    print(f"[boundary] {nx}x{ny} {prec} f {np.abs(fb - f).max():.2e} h {np.abs(hb - h).max():.2e}", flush=True)
    if prec == "fp64":
        assert np.array_equal(fb, f) and np.array_equal(hb, h)
    else:
        # deviations from the reference are below the values' own size
        assert np.abs(fb - f).max() <= 14 * 2.0 ** -24 * np.abs(f).max()
        assert np.abs(hb - h).max() <= 14 * 2.0 ** -24 * np.abs(h).max()
    eps = 64 * np.finfo(np.float64).eps  # sums of 13 values, a quotient
    rho = f.sum(2)
    ux, uy = (f * EX).sum(2) * c / rho, (f * EY).sum(2) * c / rho
    assert np.abs(m["rho"] - rho).max() <= eps * rho.max()
    scale = np.abs(f).sum(2).max() * 2 * c / rho.min()
    assert np.abs(m["ux"] - ux).max() <= eps * scale and np.abs(m["uy"] - uy).max() <= eps * scale


def test_one_array_keeps_the_other(gpu_lib):
    import ctypes as C
    from uq_amd.capi import dptr
    s = gpu_lib.Solver(_case(35, 21), "fp64")
    try:
        f0, h0 = s.get_dist()
        f, h = _values(f0, h0, 1)
        null = C.POINTER(C.c_double)()
        assert gpu_lib.lib().lbm_set_dist(s.handle, dptr(f.reshape(-1)), null) == 0
        fb, hb = s.get_dist()
        assert np.array_equal(fb, f) and np.array_equal(hb, h0)
        assert gpu_lib.lib().lbm_set_dist(s.handle, null, dptr(h.reshape(-1))) == 0
        out = np.empty(h.size)
        assert gpu_lib.lib().lbm_get_dist(s.handle, null, dptr(out)) == 0
        assert np.array_equal(out.reshape(h.shape), h)
    finally:
        s.close()


def test_copies_of_several_threads(gpu_lib):
    """Solvers read and written by four threads at once, multi-piece copies."""
    solvers = [gpu_lib.Solver(_case(300 + k, 200), "fp64") for k in range(4)]
    bad = []

    def work(k):
        s = solvers[k]
        f0, h0 = s.get_dist()
        for rep in range(3):
            f, h = _values(f0, h0, 10 * k + rep)
            s.set_dist(f, h)
            fb, hb = s.get_dist()
            if not (np.array_equal(fb, f) and np.array_equal(hb, h)):
                bad.append((k, rep))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for s in solvers:
        s.close()
    gpu_lib.release_cached()
    assert not bad
