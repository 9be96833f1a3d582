"""Solves whose input holds a number that is none: what they leave and say."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    inp = {k: np.arange(n) * 0.5 for k in ("xf", "yf", "zf")}
    for k in ("gxcf", "gycf", "gzcf"):
        inp[k] = rng.uniform(-0.1, 0.1, 4 * n * n)
    for k in ("a1cf", "a2cf", "a3cf"):
        inp[k] = rng.uniform(1.0, 2.0, n**3)
    inp["ccf"] = np.full(n**3, 0.5)
    inp["fcf"] = rng.standard_normal(n**3)
    inp["tcf"] = np.zeros(n**3)
    return inp


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("key", ["a2cf", "ccf"])
def test_operator_not_finite(mg, bad, key):
    """An operator with an inf or NaN in it: a mixed solve makes no cycle and
    leaves the boundary values around the iterate 0; an FP64 one shows NaN.
    Alone and grouped."""
    print(f"operator {key} {bad}", flush=True)
    n, nlev = 17, 3
    inp = _inputs(n, 4)
    inp[key][(8 * n + 7) * n + 9] = bad
    iparm, rparm = mg.make_params(n, nlev)
    ctxs = [mg.Context(iparm, rparm, inp) for _ in range(2)]
    for solve in (lambda m: ctxs[0].solve(m), lambda m: mg.solve_group(ctxs, m)):
        solve(mg.PMG_MIXED)
        u, st = ctxs[0].u().reshape(n, n, n), ctxs[0].stats()
        assert st["iters"] == 0 and np.isnan(st["relres"]) and len(ctxs[0].history()) == 0
        assert np.all(np.isfinite(u)) and not np.any(u[1:-1, 1:-1, 1:-1])
        assert np.array_equal(u[1:-1, 1:-1, 0].ravel(),
                              inp["gxcf"][:n * n].reshape(n, n)[1:-1, 1:-1].ravel())
        solve(mg.PMG_FP64)
        assert np.isnan(ctxs[0].u()).any() and np.isnan(ctxs[0].stats()["relres"])
    for c in ctxs:
        c.close()
