"""The kernels of 27-point levels that take pairs of i-adjacent points
(residual, product, restriction, damped prolongation, zero-start sweeps)
against the CPU oracle at the sizes where pairs, tiles and chunks end: even
and odd rows (a last pair of one point), the smallest grids, one- and
four-wavefront workgroups (1024 one-wavefront tiles is the line), chunks of
four planes with a ragged last one (100 planes and more).  Tolerance: sums of
at most 54 terms whose only difference is FMA contraction, 1e-13 of the
largest value; the damped correction also divides two dot products of n
terms summed in another order (n eps / 2 of their absolute sums), 1e-11."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

dp = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def _call(mg, name, *args):
    rc = getattr(mg.lib(), name)(*args)
    assert rc == 0, f"{name} returned {rc}"


def _level(dims, rng):
    """Random 27-point operator and two vectors with zero boundary."""
    nx, ny, nz = dims
    N = nx * ny * nz
    ac = rng.uniform(0.1, 1.0, 14 * N)
    ac[:N] += 26.0
    cc = rng.uniform(0.0, 1.0, N)
    mask = np.zeros((nz, ny, nx))
    mask[1:-1, 1:-1, 1:-1] = 1
    f, x = ((rng.standard_normal((nz, ny, nx)) * mask).ravel() for _ in range(2))
    return ac, cc, f, x


DIMS = [(3, 3, 3), (4, 3, 5), (6, 5, 4), (9, 12, 7), (66, 5, 103), (131, 66, 18), (65, 64, 12)]


@pytest.mark.parametrize("dims", DIMS)
def test_resid_matvec_27(mg, orc, dims):
    print(f"pairs resid/matvec dims={dims}", flush=True)
    rng = np.random.default_rng(sum(dims))
    ac, cc, f, x = _level(dims, rng)
    for name, mine in (("mresid", (ac, cc, f, x)), ("matvec", (ac, cc, x))):
        got, ref = np.zeros(x.size), np.zeros(x.size)
        _call(mg, "pmg_" + name, *dims, 27, *(dp(a) for a in mine), dp(got))
        getattr(orc.olib(), "pmgo_" + name)(*dims, 27, *(dp(a) for a in mine), dp(ref))
        assert _rel(got, ref) < 1e-13, name


@pytest.mark.parametrize("dc", [(3, 3, 3), (4, 3, 5), (6, 5, 4), (9, 12, 7), (33, 18, 20),
                                (80, 68, 41)])
def test_transfers(mg, orc, dc):
    """Restriction, plain and damped prolongation between a grid and the one
    of about half its size, with random weights."""
    print(f"pairs transfers coarse={dc}", flush=True)
    df = tuple(2 * v - 1 for v in dc)
    rng = np.random.default_rng(7 + sum(dc))
    Nc, Nf = np.prod(dc), np.prod(df)
    pc = rng.uniform(0.1, 1.0, 27 * Nc)
    ac, cc, w0, xc = _level(dc, rng)
    fine = rng.standard_normal(Nf)
    got, ref = np.zeros(Nc), np.zeros(Nc)
    _call(mg, "pmg_restrc", *df, *dc, dp(fine), dp(got), dp(pc))
    orc.olib().pmgo_restrc(*df, *dc, dp(fine), dp(ref), dp(pc))
    assert _rel(got, ref) < 1e-13
    got, pxc = np.zeros(Nf), np.zeros(Nf)
    _call(mg, "pmg_interp", *dc, *df, dp(xc), dp(got), dp(pc))
    orc.olib().pmgo_interp(*dc, *df, dp(xc), dp(pxc), dp(pc))
    assert _rel(got, pxc) < 1e-13
    # xf(interior) += (xc . w0) / (xc . A xc) P xc; the boundary stays as it is
    y = np.zeros(Nc)
    orc.olib().pmgo_matvec(*dc, 27, dp(ac), dp(cc), dp(xc), dp(y))
    ref = fine.copy()
    inner = np.zeros(df[::-1], bool)
    inner[1:-1, 1:-1, 1:-1] = True
    ref[inner.ravel()] += (xc @ w0) / (xc @ y) * pxc[inner.ravel()]
    got = fine.copy()
    _call(mg, "pmg_correct", *dc, *df, 27, dp(ac), dp(cc), dp(xc), dp(w0), dp(pc), dp(got))
    assert np.array_equal(got[~inner.ravel()], fine[~inner.ravel()])
    assert _rel(got, ref) < 1e-11


@pytest.mark.parametrize("iadj", [0, 1])
@pytest.mark.parametrize("dims", [(4, 5, 6), (33, 25, 19), (80, 21, 9), (140, 9, 8)])
def test_gsrb_zero_27(mg, orc, dims, iadj):
    """Zero-start sweeps (their first half does not load the planes above and
    below): one, two and three of them from an array whose interior is not
    zero."""
    print(f"pairs gsrb_zero dims={dims} iadjoint={iadj}", flush=True)
    rng = np.random.default_rng(sum(dims) + iadj)
    ac, cc, f, x = _level(dims, rng)
    for sweeps in (1, 2, 3):
        got = x.copy()
        _call(mg, "pmg_gsrb_zero", *dims, 27, dp(ac), dp(cc), dp(f), dp(got), sweeps, iadj)
        ref = orc.gsrb(0, 27, ac, cc, f, np.zeros(x.size), sweeps, iadj, dims=dims)
        assert _rel(got, ref) < 1e-12, sweeps
