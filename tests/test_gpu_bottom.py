"""The two coarsest levels of a cycle as the bottom kernels run them
(pmg_bottom.hip), on boxes with three different sides: against the CPU
oracle's solve with the same cycle count (FP64 to 1e-10 of the largest
potential, the bar of every FP64 solve here; mixed precision to 1e-6), alone
and grouped with the same bits.  The level above the coarsest is 9 x 13 x 11
(both precisions take the kernels), 5^3 over a single unknown, 17^3 (FP32
only) and 17 x 25 x 21 (neither); sweep counts of 0 to 3, odd ones among
them.  Two-level grids over 11^3 and 13^3 take the coarsest CG with three
points per thread, in workgroups of up to 256 threads and beyond."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(dims, seed):
    nx, ny, nz = dims
    N = nx * ny * nz
    rng = np.random.default_rng(seed)
    inp = {k: np.arange(n) * 0.5 for k, n in zip(("xf", "yf", "zf"), dims)}
    for k, n in (("gxcf", ny * nz), ("gycf", nx * nz), ("gzcf", nx * ny)):
        inp[k] = rng.uniform(-0.1, 0.1, 4 * n)
    eps = np.where(rng.random(N) < 0.3, 2.0, 78.54)
    for k in ("a1cf", "a2cf", "a3cf"):
        inp[k] = eps * rng.uniform(0.5, 1.0, N)
    inp["ccf"] = np.where(rng.random(N) < 0.5, 0.0, 0.8)
    inp["fcf"] = rng.standard_normal(N)
    inp["tcf"] = np.zeros(N)
    return inp


KEYS = ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf", "a3cf", "ccf", "fcf", "tcf")


@pytest.mark.parametrize("dims,nlev,nu", [((17, 25, 21), 3, (2, 2)), ((33, 49, 41), 4, (1, 3)),
                                          ((17, 17, 17), 4, (2, 2)), ((33, 33, 33), 3, (3, 1)),
                                          ((33, 49, 41), 3, (2, 2)), ((17, 25, 21), 3, (0, 2)),
                                          ((21, 21, 21), 2, (2, 2)), ((25, 25, 25), 2, (2, 2))])
def test_bottom_levels(mg, orc, dims, nlev, nu):
    print(f"bottom dims={dims} nlev={nlev} nu={nu}", flush=True)
    inp = _inputs(dims, sum(dims) + nlev)
    sz = mg.Vmgsz(2, 0, 0, *dims, nlev)
    iparm, rparm = mg.Vpackmg(sz["iretot"], sz["iintot"], *dims, nlev, nu1=nu[0], nu2=nu[1])

    def solve(fn):
        u = np.zeros(dims[0] * dims[1] * dims[2])
        a = [inp[k].copy() for k in KEYS]
        rc = fn(iparm.copy(), rparm.copy(), np.zeros(sz["iintot"], np.int32),
                np.zeros(sz["iretot"]), u, *a)
        assert rc == 0
        return u

    ref = solve(orc.mgdriv)
    its = orc.last_stats()[0]
    u = solve(mg.Vmgdriv)
    assert mg.last_stats()[0] == its
    assert np.max(np.abs(u - ref)) <= 1e-10 * np.max(np.abs(ref))
    ctxs = [mg.Context(iparm, rparm, inp) for _ in range(2)]
    for mode, tol in ((mg.PMG_FP64, 1e-10), (mg.PMG_MIXED, 1e-6)):
        ctxs[0].solve(mode)
        alone = ctxs[0].u()
        assert np.max(np.abs(alone - ref)) <= tol * np.max(np.abs(ref))
        mg.solve_group(ctxs, mode)
        assert np.array_equal(ctxs[0].u(), alone) and np.array_equal(ctxs[1].u(), alone)
    for c in ctxs:
        c.close()
