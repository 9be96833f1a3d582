"""Boundary potentials on the GPU (k_pb_faces) where its staging can go wrong:
uncharged atoms first, last, all or none, chunks of 256 atoms with one more
or one less, against the CPU oracle, to 1e-13 of the largest (the bar of the
faces); and an atom so far away that its term underflows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,zeros", [(1, "none"), (1, "all"), (255, "none"), (256, "first"),
                                          (257, "last"), (300, "mixed"), (513, "all but one"),
                                          (40, "far")])
def test_faces_staging(mg, orc, natoms, zeros):
    print(f"faces natoms={natoms} zeros={zeros}", flush=True)
    n, h = 17, 1.5
    rng = np.random.default_rng(natoms)
    at = np.column_stack([rng.uniform(-8, 8, (natoms, 3)), rng.uniform(1.2, 2.0, natoms),
                          rng.choice([-1.0, 0.5, 1.0], natoms)])
    if zeros == "all":
        at[:, 4] = 0.0
    elif zeros == "first":
        at[:200, 4] = 0.0
    elif zeros == "last":
        at[56:, 4] = 0.0
    elif zeros == "mixed":
        at[rng.random(natoms) < 0.5, 4] = 0.0
    elif zeros == "all but one":
        at[np.arange(natoms) != 511, 4] = 0.0
    elif zeros == "far":
        at[7, :3] = 1e9, -1e9, 1e9
    want = orc.pbe_assemble(n, h, 0.15, at)
    got = mg.pbe_assemble(n, h, 0.15, at)
    for k in ("gxcf", "gycf", "gzcf"):
        assert np.max(np.abs(got[k] - want[k])) <= 1e-13 * np.max(np.abs(want[k])), k
