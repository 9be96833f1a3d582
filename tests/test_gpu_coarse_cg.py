"""The coarsest CG on the unit-diagonal operator (k_cg_rows of FP64 cycles),
which ends when its solution has settled: two-level solves against the CPU
oracle's, whose coarsest CG runs its 100 iterations, with the same cycle
count and to 1e-10 of the largest potential (the bar of every FP64 solve
here).  Coarsest levels of one unknown to 11^3 unknowns, two and three
points per thread, ragged rows; coefficients over one and (where 100 plain
iterations settle too) over four decades, within and beyond the span of the
diagonal that takes the scaled form; and a zero right-hand side, whose coarse solution is zero (damping 0)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf", "a3cf", "ccf", "fcf", "tcf")


@pytest.mark.parametrize("dims,low", [((5, 5, 5), 2.0), ((9, 7, 11), 2.0), ((17, 17, 17), 2.0),
                                      ((21, 21, 21), 2.0), ((25, 21, 23), 2.0),
                                      ((25, 25, 25), 2.0), ((5, 5, 5), 0.01),
                                      ((9, 7, 11), 0.01)])
def test_two_levels(mg, orc, dims, low):
    print(f"coarse cg dims={dims} low={low}", flush=True)
    nx, ny, nz = dims
    N = nx * ny * nz
    rng = np.random.default_rng(11)
    inp = {k: np.arange(n) * 0.5 for k, n in zip(("xf", "yf", "zf"), dims)}
    for k, n in (("gxcf", ny * nz), ("gycf", nx * nz), ("gzcf", nx * ny)):
        inp[k] = rng.uniform(-0.1, 0.1, 4 * n)
    k, j, i = np.meshgrid(*(np.linspace(-1, 1, n) for n in (nz, ny, nx)), indexing="ij")
    eps = np.where(i * i + j * j + k * k < 0.4, low, 78.54).ravel()
    for a in ("a1cf", "a2cf", "a3cf"):
        inp[a] = eps.copy()
    inp["ccf"] = np.where(eps == low, 0.0, 0.8)
    inp["fcf"] = rng.standard_normal(N)
    inp["tcf"] = np.zeros(N)
    sz = mg.Vmgsz(2, 0, 0, nx, ny, nz, 2)
    got = []
    for zero in (False, True):
        if zero:
            inp["fcf"][:] = 0.0
            for g in ("gxcf", "gycf", "gzcf"):
                inp[g][:] = 0.0
        for drv, stats in ((mg.Vmgdriv, mg.last_stats), (orc.mgdriv, orc.last_stats)):
            iparm, rparm = mg.Vpackmg(sz["iretot"], sz["iintot"], nx, ny, nz, 2)
            u = np.zeros(N)
            drv(iparm, rparm, np.zeros(sz["iintot"], np.int32), np.zeros(sz["iretot"]), u,
                *(inp[q].copy() for q in KEYS))
            got.append((u, stats()[0]))
        (ug, ig), (uo, io) = got[-2:]
        if zero:
            assert not np.any(ug) and not np.any(uo)
        else:
            assert ig == io
            assert np.max(np.abs(ug - uo)) <= 1e-10 * np.max(np.abs(uo))
