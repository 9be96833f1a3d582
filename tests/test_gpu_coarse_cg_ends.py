"""The coarsest CG (k_cg_rows) where its residual norm leaves the middle of
the range: one FP64 cycle on two levels against the CPU oracle's, to 1e-10 of
the largest potential (the bar of every FP64 solve here)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf", "a3cf", "ccf", "fcf", "tcf")


def _cycle(mg, orc, dims, f):
    nx, ny, nz = dims
    N = nx * ny * nz
    inp = {k: np.arange(n) * 0.5 for k, n in zip(("xf", "yf", "zf"), dims)}
    for k, n in (("gxcf", ny * nz), ("gycf", nx * nz), ("gzcf", nx * ny)):
        inp[k] = np.zeros(4 * n)
    for k in ("a1cf", "a2cf", "a3cf"):
        inp[k] = np.ones(N)
    inp["ccf"], inp["fcf"], inp["tcf"] = np.full(N, 0.1), f.ravel().copy(), np.zeros(N)
    sz = mg.Vmgsz(2, 0, 0, nx, ny, nz, 2)
    out = []
    for drv in (mg.Vmgdriv, orc.mgdriv):
        iparm, rparm = mg.Vpackmg(sz["iretot"], sz["iintot"], nx, ny, nz, 2, itmax=1)
        u = np.zeros(N)
        drv(iparm, rparm, np.zeros(sz["iintot"], np.int32), np.zeros(sz["iretot"]), u,
            *(inp[k].copy() for k in KEYS))
        out.append(u)
    return out


# Coarse levels of 2 x 1 x 1 and 2 x 2 x 2 unknowns in a uniform medium: a
# right-hand side even in x but for a small odd part is almost an eigenvector
# of the coarse operator, and its first iteration leaves that part alone.
@pytest.mark.parametrize("dims", [(7, 5, 5), (7, 7, 7)])
def test_almost_an_eigenvector(mg, orc, dims):
    print(f"coarse cg almost an eigenvector dims={dims}", flush=True)
    nx, ny, nz = dims
    f = np.zeros((nz, ny, nx))
    f[1:-1, 1:-1, 1:-1] = 1.0
    odd = np.broadcast_to(np.linspace(-1.0, 1.0, nx), f.shape) * f
    for e in np.geomspace(3e-8, 3e-10, 24):
        got, want = _cycle(mg, orc, dims, f + e * odd)
        assert np.max(np.abs(got - want)) <= 1e-10 * np.max(np.abs(want)), e


# coarse levels of 3^3 and 5^3 unknowns
@pytest.mark.parametrize("dims", [(9, 9, 9), (13, 13, 13)])
@pytest.mark.parametrize("scale", [1e120, 1e200])
def test_overflow(mg, orc, dims, scale):
    """A right-hand side whose square overflows shows as it does in the
    oracle; one whose square does not is solved."""
    print(f"coarse cg overflow dims={dims} scale={scale}", flush=True)
    nx, ny, nz = dims
    f = np.random.default_rng(3).standard_normal((nz, ny, nx)) * scale
    got, want = _cycle(mg, orc, dims, f)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.max(np.abs(got - want)[ok]) <= 1e-10 * np.max(np.abs(want[ok]))
