"""Results in the caller's host memory: the copies through the pinned pieces
(pmg_hostcopy.hip) hold the same bytes as the runtime's own copy, which a
pinned destination takes, on grids below the smallest copy that is cut
(65^3), with a remainder of a piece, of fewer pieces than slots and of more
(161^3: 16 full pieces and one more; 193^3: 28), and from three threads at
once (two pinned rings); the drivers' rwork is written or zeroed everywhere."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("n,nlev", [(65, 4), (81, 4), (97, 5), (145, 5), (161, 5), (193, 6)])
def test_potential_pageable_and_pinned(mg, n, nlev):
    print(f"host copy n={n}", flush=True)
    iparm, rparm = mg.make_params(n, nlev)
    ctx = mg.Context(iparm, rparm, pbe=(0.5, 0.15, mg.pbe_molecule(100, 12.0, 0, 3)))
    ctx.solve(mg.PMG_FP64)
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime the library uses
    pinned = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(8 * n ** 3), 0) == 0
    assert mg.lib().pmg_ctx_get_u(ctx._h, ctypes.cast(pinned, D)) == 0
    want = np.ctypeslib.as_array(ctypes.cast(pinned, D), (n ** 3,)).copy()
    assert hip.hipHostFree(pinned) == 0
    assert np.any(want != 0.0)
    odd = np.full(n ** 3 + 3, np.nan)  # not page aligned, neighbours kept
    assert mg.lib().pmg_ctx_get_u(ctx._h, odd[1:].ctypes.data_as(D)) == 0
    assert np.array_equal(odd[1:-2], want)
    assert np.isnan(odd[0]) and np.all(np.isnan(odd[-2:]))
    got = [None] * 3

    def fetch(q):
        got[q] = ctx_q[q].u()

    ctx_q = [ctx] + [mg.Context(iparm, rparm, pbe=(0.5, 0.15, mg.pbe_molecule(100, 12.0, 0, 3)))
                     for _ in range(2)]
    for c in ctx_q[1:]:
        c.solve(mg.PMG_FP64)
    th = [threading.Thread(target=fetch, args=(q,)) for q in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(np.array_equal(g, want) for g in got)


@pytest.mark.parametrize("nonlin", [0, 1])
@pytest.mark.parametrize("n,nlev", [(33, 3), (65, 4)])
def test_driver_work_array(mg, orc, n, nlev, nonlin):
    print(f"rwork n={n} nonlin={nonlin}", flush=True)
    mg.Vmypdefinitnpbe(2, [1.0, -1.0], [0.5, 0.5])
    inp = orc.pbe_assemble(n, 0.5, 0.15, mg.pbe_molecule(40, 6.0, 0, 7))
    iparm, rparm = mg.make_params(n, nlev, nonlin=nonlin)
    sz = mg.Vmgsz(2, 0, 0, n, n, n, nlev)
    nf, narr, narrc, nrpc = (sz[k] for k in ("nf", "narr", "narrc", "n_rpc"))
    gap = 2 * nf if nonlin else 0
    total = sz["iretot"] + gap
    rw = np.full(total + 5, np.nan)
    u = np.zeros(n ** 3)
    (mg.Vnewdriv if nonlin else mg.Vmgdriv)(
        iparm, rparm, np.zeros(sz["iintot"], np.int32), rw, u,
        *(inp[k].copy() for k in ("xf", "yf", "zf", "gxcf", "gycf", "gzcf", "a1cf", "a2cf",
                                  "a3cf", "ccf", "fcf", "tcf")))
    assert np.all(np.isnan(rw[total:])) and not np.any(np.isnan(rw[:total]))
    ctx = mg.Context(iparm, rparm, inp)
    lev = [ctx.level(q + 1) for q in range(nlev)]
    cc, fc = (np.concatenate([l[q] for l in lev]) for q in (1, 2))
    pc = np.concatenate([l[3] for l in lev[:-1]])
    ac = np.concatenate([l[0] for l in lev])
    want = np.zeros(total)
    o = nrpc
    want[o:o + cc.size] = cc
    o += narr
    want[o:o + fc.size] = fc
    o += narr + gap
    want[o:o + pc.size] = pc
    o += 27 * narrc
    want[o:o + ac.size] = ac
    assert np.array_equal(rw[:total], want)
