"""The bottom kernels (pmg_bottom.hip) on the paths that enter them besides
the linear solve: the class-style PCG (forward sweeps on the way up, a
warm-started coarsest CG with its damping factor) and Newton (the Jacobian's
term as the diagonal's second part), in both precisions, on levels of 13^3
and 9 x 13 x 11 above the coarsest; against the CPU oracle with the same
iterations, to the bars of tests/test_gpu_pcg.py and test_gpu_parity.py.
The rule that sends a level there is looked at by itself (on the CPU)."""
import ctypes

import numpy as np
import pytest

CASES = [((49, 49, 49), 4), ((33, 49, 41), 4)]
KEYS = ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf", "a3cf", "ccf", "fcf", "tcf")


def _taken(mg, level, precision, numdia=27, numdiac=27, coarse=None):
    fn = getattr(mg.lib(), f"_ZN3pmg11bottom_fitsI{precision}EEbRKNS_3DimEiS3_i")
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.POINTER(ctypes.c_int), ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                   ctypes.c_int]
    coarse = coarse or tuple((n - 1) // 2 + 1 for n in level)
    return fn((ctypes.c_int * 3)(*level), numdia, (ctypes.c_int * 3)(*coarse), numdiac)


def _second_coarsest(dims, nlev):
    return tuple((n - 1) // (1 << (nlev - 2)) + 1 for n in dims)


def test_rule(mg):
    for level, f, d in [((13, 13, 13), True, True), ((9, 13, 11), True, True),
                        ((5, 5, 5), True, True), ((17, 17, 17), True, False),
                        ((17, 17, 19), False, False), ((21, 21, 21), False, False),
                        ((5, 5, 129), True, False), ((3, 5, 5), False, False)]:
        assert _taken(mg, level, "f") == f and _taken(mg, level, "d") == d, level
    assert not _taken(mg, (13, 13, 13), "d", numdia=7)
    assert not _taken(mg, (13, 13, 13), "d", numdiac=7)
    assert not _taken(mg, (13, 13, 13), "f", coarse=(7, 7, 6))
    for dims, nlev in CASES:  # what the tests below rely on
        assert _taken(mg, _second_coarsest(dims, nlev), "f")
        assert _taken(mg, _second_coarsest(dims, nlev), "d")


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


def _oracle(orc, mg, fn, inp, iparm, rparm, dims, nlev, *more):
    sz = mg.Vmgsz(2, 0, 0, *dims, nlev)
    u = np.zeros(dims[0] * dims[1] * dims[2])
    rc = fn(orc.ip(iparm), orc.dp(rparm), orc.ip(np.zeros(sz["iintot"], np.int32)),
            orc.dp(np.zeros(int(iparm[0]))), orc.dp(u),
            *(orc.dp(inp[k].copy()) for k in KEYS), *more)
    assert rc == 0
    return u, orc.last_stats()[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dims,nlev", CASES)
def test_pcg(mg, orc, dims, nlev):
    print(f"bottom pcg dims={dims}", flush=True)
    inp = _inputs(dims, 21)
    sz = mg.Vmgsz(2, 0, 0, *dims, nlev)
    iparm, rparm = mg.Vpackmg(sz["iretot"], sz["iintot"], *dims, nlev)
    ref, its = _oracle(orc, mg, orc.olib().pmgo_pcgdriv, inp, iparm, rparm, dims, nlev, 0)
    ctx = mg.Context(iparm, rparm, inp)
    for mode, tol in ((mg.PMG_FP64, 1e-10), (mg.PMG_MIXED, 1e-6)):
        ctx.pcg(mode)
        if mode == mg.PMG_FP64:
            assert ctx.stats()["iters"] == its
        assert np.max(np.abs(ctx.u() - ref)) <= tol * np.max(np.abs(ref))
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("mgkey", [0, 1])
@pytest.mark.parametrize("dims,nlev", CASES)
def test_newton(mg, orc, dims, nlev, mgkey):
    print(f"bottom newton dims={dims} mgkey={mgkey}", flush=True)
    ions = ([1.0, -1.0], [0.5, 0.5])
    mg.Vmypdefinitnpbe(2, *ions)
    orc.mypdefinit(*ions)
    inp = _inputs(dims, 22)
    sz = mg.Vmgsz(2, 0, 0, *dims, nlev)
    nf = dims[0] * dims[1] * dims[2]
    iparm, rparm = mg.Vpackmg(sz["iretot"] + 2 * nf, sz["iintot"], *dims, nlev, nonlin=1,
                              errtol=1e-8, mgkey=mgkey)
    ref, its = _oracle(orc, mg, orc.olib().pmgo_newdriv, inp, iparm, rparm, dims, nlev)
    ctx = mg.Context(iparm, rparm, inp)
    for mode, tol in ((mg.PMG_FP64, 1e-9), (mg.PMG_MIXED, 1e-6)):
        ctx.solve(mode)
        if mode == mg.PMG_FP64:
            assert ctx.stats()["iters"] == its
        assert np.max(np.abs(ctx.u() - ref)) <= tol * np.max(np.abs(ref))
    ctx.close()
