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


FACES = ("gxcf", "gycf", "gzcf")


def _atoms(natoms, seed):
    rng = np.random.default_rng(seed)
    return np.column_stack([rng.uniform(-8, 8, (natoms, 3)), rng.uniform(1.2, 2.0, natoms),
                            rng.choice([-1.0, 0.5, 1.0], natoms)])


@pytest.mark.parametrize("field", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("charge", [1.0, 0.0])
def test_faces_nan(mg, orc, field, charge):
    """A record that is no number shows in every boundary value, as in the
    oracle, whether or not the atom carries a charge."""
    print(f"faces nan field={field} charge={charge}", flush=True)
    at = _atoms(300, field)
    at[270, 4] = charge
    at[270, field] = np.nan
    want = orc.pbe_assemble(17, 1.5, 0.15, at)
    got = mg.pbe_assemble(17, 1.5, 0.15, at)
    for k in FACES:
        assert np.array_equal(np.isnan(got[k]), np.isnan(want[k])), k
        assert np.isnan(got[k]).any(), k


@pytest.mark.parametrize("natoms", [3, 255, 256, 257, 511])
def test_faces_uncharged(mg, natoms):
    """Uncharged atoms change no bit of the sums: as charges too small to
    show they give the same faces."""
    print(f"faces uncharged natoms={natoms}", flush=True)
    at = _atoms(natoms, natoms)
    none = np.random.default_rng(1).random(natoms) < 0.4
    got = []
    for q in (0.0, 1e-290):
        at[none, 4] = q
        got.append(mg.pbe_assemble(17, 1.5, 0.15, at))
    for k in FACES:
        assert np.array_equal(got[0][k], got[1][k]), k
