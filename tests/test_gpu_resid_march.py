"""The marching residual without the precomputed diagonal (the residual
entry points on caller arrays) against numpy in FP64: boxes whose tiles are
ragged in i and j and whose last k chunk is short, one tile wide, and one
the column kernel keeps.  FP64 sums of seven terms: 16 roundings of the
largest term, then the FP32 store's half ulp."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

_D = ctypes.POINTER(ctypes.c_double)
_F = ctypes.POINTER(ctypes.c_float)


@pytest.mark.parametrize("dims", [(113, 177, 161), (161, 97, 193), (61, 200, 199), (20, 183, 200),
                                  (129, 65, 33)])
def test_resid_march(mg, dims):
    print(f"resid march dims={dims}", flush=True)
    nx, ny, nz = dims
    rng = np.random.default_rng(3)
    ac = rng.uniform(0.1, 2.0, (4, nz, ny, nx))
    cc, f, x = (rng.standard_normal((nz, ny, nx)) for _ in range(3))
    r = np.full((nz, ny, nx), np.nan, np.float32)
    l1 = ctypes.c_double()
    rc = mg.lib().pmg_mresid_mixed(nx, ny, nz, ac.ctypes.data_as(_D), cc.ctypes.data_as(_D),
                                   f.ctypes.data_as(_D), x.ctypes.data_as(_D),
                                   r.ctypes.data_as(_F), ctypes.byref(l1))
    assert rc == 0
    want, size = f - (ac[0] + cc) * x, np.abs(f) + np.abs((ac[0] + cc) * x)
    for p, d in ((1, 2), (2, 1), (3, 0)):
        up, dn = ac[p] * np.roll(x, -1, d), np.roll(ac[p], 1, d) * np.roll(x, 1, d)
        want += up + dn
        size += np.abs(up) + np.abs(dn)
    inner = (slice(1, -1),) * 3
    assert np.isnan(r).sum() == r.size - r[inner].size  # the boundary is left as given
    err = np.abs(r[inner].astype(np.float64) - want[inner])
    assert np.all(err <= 2.0 ** -24 * np.abs(want[inner]) + 16 * 2.0 ** -53 * size[inner])
    total = np.abs(want[inner]).sum()
    assert abs(l1.value - total) <= 1e-12 * total
