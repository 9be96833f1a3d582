"""The class-style PCG where its fine product and residuals march (two
62-column tiles across i and ragged ones in j, k chunks of 18 planes and a
short last one) on a box with three different sides, against the CPU
oracle: the same iterations, FP64 potential to 1e-10 of the largest (the bar
of every FP64 solve here), to the tolerance and counted; the iteration it
stops at makes no further direction."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf", "a3cf", "ccf", "fcf", "tcf")


@pytest.mark.parametrize("num_iters", [0, 1, 2])
def test_pcg_march(mg, orc, num_iters):
    dims, nlev = (113, 177, 161), 5
    print(f"pcg march dims={dims} num_iters={num_iters}", flush=True)
    nx, ny, nz = dims
    N = nx * ny * nz
    rng = np.random.default_rng(5)
    inp = {k: np.arange(n) * 0.5 for k, n in zip(("xf", "yf", "zf"), dims)}
    for k, n in (("gxcf", ny * nz), ("gycf", nx * nz), ("gzcf", nx * ny)):
        inp[k] = rng.uniform(-0.1, 0.1, 4 * n)
    eps = np.where(rng.random(N) < 0.3, 2.0, 78.54)
    for k in ("a1cf", "a2cf", "a3cf"):
        inp[k] = eps * rng.uniform(0.5, 1.0, N)
    inp["ccf"] = np.where(rng.random(N) < 0.5, 0.0, 0.8)
    inp["fcf"] = rng.standard_normal(N)
    inp["tcf"] = np.zeros(N)
    sz = mg.Vmgsz(2, 0, 0, *dims, nlev)
    iparm, rparm = mg.Vpackmg(sz["iretot"], sz["iintot"], *dims, nlev)
    ctx = mg.Context(iparm, rparm, inp)
    ctx.pcg(mg.PMG_FP64, num_iters)
    u, its = ctx.u(), ctx.stats()["iters"]
    ctx.close()
    ref = np.zeros(N)
    a = [inp[k].copy() for k in KEYS]
    rc = orc.olib().pmgo_pcgdriv(orc.ip(iparm), orc.dp(rparm),
                                 orc.ip(np.zeros(sz["iintot"], np.int32)),
                                 orc.dp(np.zeros(sz["iretot"])), orc.dp(ref),
                                 *(orc.dp(v) for v in a), num_iters)
    assert rc == 0 and its == orc.last_stats()[0]
    assert num_iters == 0 or its == num_iters
    assert np.max(np.abs(u - ref)) <= 1e-10 * np.max(np.abs(ref))
