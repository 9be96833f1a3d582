"""The FP32 cycle's arithmetic to the bit.

The coarsest CG of a mixed cycle stops at a relative 1e-2, after up to 30
iterations where the coarse diagonal spans a factor of hundreds; by then its
iterates have grown one changed rounding of their right-hand side far enough
to change the iteration count, and with it the potential by up to 1e-9 of
its norm.  So the order of every sum, and which product of two the
multiply-add rounds, is part of a mixed solve's result: these tests restate
both and allow no difference.

`fma32` rounds once (the exact product and sum, rounded to odd in 64 bits
first); the FP64 multiply-add is the C library's."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = np.float32
_F = ctypes.POINTER(ctypes.c_float)
_D = ctypes.POINTER(ctypes.c_double)
_libm = ctypes.CDLL("libm.so.6")
_libm.fma.restype = ctypes.c_double
_libm.fma.argtypes = [ctypes.c_double] * 3
_fma = np.frompyfunc(_libm.fma, 3, 1)


def fma64(a, b, c):
    return np.asarray(_fma(a, b, c), np.float64)


def fma32(a, b, c):
    p = a.astype(np.float64) * b.astype(np.float64)  # exact
    c = np.broadcast_to(np.asarray(c, np.float64), p.shape)
    s = np.ascontiguousarray(p + c)
    t = s - p
    e = (p - (s - t)) + (c - t)
    bits = s.view(np.int64).copy()
    odd = (bits - ((e < 0) != (s < 0))) | 1
    return np.where(e != 0, odd, bits).view(np.float64).astype(F32)


# the 26 terms: offset, plane, and whether the coupling is stored at the
# neighbour; 0-7 in the plane, 8-16 above, 17-25 below
_XY = [(0, 0), (0, 1), (0, -1), (1, 0), (-1, 0), (1, 1), (-1, 1), (1, -1), (-1, -1)]
TERMS = ([((0, 1, 0), 2, 0), ((0, -1, 0), 2, 1), ((1, 0, 0), 1, 0), ((-1, 0, 0), 1, 1),
          ((1, 1, 0), 4, 0), ((-1, 1, 0), 5, 0), ((1, -1, 0), 5, 1), ((-1, -1, 0), 4, 1)]
         + [((dx, dy, 1), pl, 0) for (dx, dy), pl in zip(_XY, (3, 8, 9, 6, 7, 10, 11, 12, 13))]
         + [((dx, dy, -1), pl, 1) for (dx, dy), pl in zip(_XY, (3, 9, 8, 7, 6, 13, 12, 11, 10))])


def fp(a):
    assert a.dtype == F32 and a.flags.c_contiguous
    return a.ctypes.data_as(_F)


def _call(mg, name, *args):
    rc = getattr(mg.lib(), name)(*args)
    assert rc == 0, f"{name} returned {rc}"


def _sweep(ac, cc, f, x, adj):
    """One 8-colour sweep of a 27-point level, arrays indexed [k, j, i]."""
    nz, ny, nx = x.shape
    colours = [(k, j, i) for k in (0, 1) for j in (0, 1) for i in (0, 1)]
    for pk, pj, pi in (colours[::-1] if adj else colours):
        kk, jj, ii = np.meshgrid(np.arange(1 + pk, nz - 1, 2), np.arange(1 + pj, ny - 1, 2),
                                 np.arange(1 + pi, nx - 1, 2), indexing="ij")

        def term(t):
            (dx, dy, dz), pl, at = t
            n = kk + dz, jj + dy, ii + dx
            return (ac[(pl,) + n] if at else ac[pl, kk, jj, ii]), x[n]

        def total(lo, hi):
            (c0, x0), (c1, x1) = term(TERMS[lo]), term(TERMS[lo + 1])
            s = fma32(c0, x0, c1 * x1)
            for t in TERMS[lo + 2:hi]:
                s = fma32(*term(t), s)
            return s

        s = f[kk, jj, ii] + ((total(0, 8) + total(8, 17)) + total(17, 26))
        x[kk, jj, ii] = s / (ac[0, kk, jj, ii] + cc[kk, jj, ii])


# rows of one, two and four pairs of points per lane, odd and even
@pytest.mark.parametrize("dims", [(9, 9, 9), (8, 5, 6), (131, 5, 7), (260, 6, 5), (3, 3, 3)])
@pytest.mark.parametrize("adj", [0, 1])
def test_sweep27(mg, dims, adj):
    print(f"sweep bits dims={dims} adj={adj}", flush=True)
    nx, ny, nz = dims
    rng = np.random.default_rng(sum(dims))
    ac = rng.uniform(0.2, 1.0, (14, nz, ny, nx)).astype(F32)
    ac[0] += F32(30)
    cc = rng.uniform(0.0, 0.1, (nz, ny, nx)).astype(F32)
    f, x = (rng.standard_normal((nz, ny, nx)).astype(F32) for _ in range(2))
    got = x.copy()
    _call(mg, "pmg_gsrb_f32", nx, ny, nz, 27, fp(ac), fp(cc), fp(f), fp(got), 1, adj, 0)
    want = x.copy()
    _sweep(ac, cc, f, want, adj)
    assert np.array_equal(got, want)
