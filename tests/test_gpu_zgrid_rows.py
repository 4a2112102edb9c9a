"""GPU: z-grid samples taken from stored rows, at the edges of the rule that decides them.

Molecules that stop at each element, in the lens or not at all; starts on, before and beyond the grid; grids
that fall on faces, on the lens's steps and on zero-length apertures; counts around a wavefront, a slice of
the workspace and the fewest that take more than one kernel; sample counts around the fewest that do; and molecules they leave to the one-kernel form
(standing, moving backwards, slow, not finite).  Every sample is that of the oracle's sampling of the molecule's
own recorded rows, in both layouts.  A molecule that starts beyond its first element goes back to it first: the
device decides a sample from the first row at or beyond its z after the first one, where the oracle searches all
rows for that z, so the expected samples of such a molecule are that rule's, restated here.
"""
import numpy as np
import pytest

from oracle import oracle as O
from trajectories import configs
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens, FieldPlates, RectangularAperture
from trajectories.engine import Engine

pytestmark = pytest.mark.gpu


def beamline(field, length=0.1, dt=configs.LENS_DT, plates=False):
    els = [CircularAperture("A", 0.3, 0.0, d=12e-3),
           ElectrostaticLens("ES lens", 0.5, length, d=2 * configs.LENS_R, V=25e3, stark=configs.stark_table(),
                             field=field, integrator="rk4", dt=dt),
           CircularAperture("B", 0.75, 0.0, d=6e-3)]
    if plates:
        els += [RectangularAperture("R", 0.8, 0.01, w=8e-3, h=8e-3),
                FieldPlates("P", 0.85, 0.1, w=6e-3)]
    return Beamline(els, 9.81)


def molecules(n, seed, odd=True):
    rs = np.random.RandomState(seed)
    X = np.vstack([rs.normal(0, configs.SIGMA_X / 2, (2, n)), rs.choice([0.0, 0.0, 0.1, -0.05, 0.3, 0.5], n)])
    V = np.vstack([rs.normal(0, configs.SIGMA_V / 4, (2, n)), rs.normal(configs.VZ_MEAN, configs.VZ_SIGMA, n)])
    if odd:
        k = rs.permutation(n)[: max(1, n // 20)]
        V[2, k] = rs.choice([0.0, -100.0, 1.0, 1e9, np.inf, np.nan, -0.0], k.size)
        V[0, k[::5]] = np.nan
        X[2, k[::7]] = np.nan
    return X, V


def in_one_pass(rows, z_start, z_step, n):
    """The device's rule (a sample before the first row takes the last row) on rows of any order."""
    out = np.full((n, 6), np.nan)
    z, last = rows[:, 2], rows[-1, 2]

    def ahead(r, zk):
        x, y, z0, vx, vy, vz, ax, ay, az, t = rows[r]
        dt = (zk - z0) / vz
        dt2 = dt * dt
        return ((x + vx * dt) + (ax * dt2) / 2.0, (y + vy * dt) + (ay * dt2) / 2.0, vx + ax * dt, vy + ay * dt,
                vz + az * dt, t + dt)

    for i in range(n):
        zk = z_start + i * z_step
        if zk < z[0]:
            if not last < zk:
                out[i] = ahead(len(rows) - 1, zk)
        elif not zk > last:
            r = 0 if zk == z[0] else next((r for r in range(1, len(rows)) if z[r] >= zk), None)
            if r is None:
                continue
            if z[r] != zk and r + 1 < len(rows) and z[r + 1] == zk:
                r += 1
            out[i] = rows[r, [0, 1, 3, 4, 5, 9]] if z[r] == zk else ahead(r - 1, zk)
    return out


def check(eng, X, V, z_start, z_step, n_samples, js, **kw):
    field, w1, l1 = eng.zgrid(*X, *V, z_start=z_start, z_step=z_step, n_samples=n_samples, **kw)
    by_mol, w2, l2 = eng.zgrid_by_molecule(*X, *V, z_start=z_start, z_step=z_step, n_samples=n_samples, **kw)
    assert np.array_equal(w1, w2) and np.array_equal(l1, l2)
    assert np.array_equal(field.transpose(2, 1, 0), by_mol, equal_nan=True)
    sub = {k: v[js] for k, v in kw.items()}
    rows, n_rows, lab = eng.record_rows(*X[:, js], *V[:, js], **sub)
    assert np.array_equal(lab, l1[js])
    for q, j in enumerate(js):
        own = rows[q][: n_rows[q]]
        if (np.diff(own[:, 2]) < 0).any():
            with np.errstate(all="ignore"):
                want = in_one_pass(own, z_start, z_step, n_samples)
        else:
            want = O.zgrid_from_rows(rows[q], int(n_rows[q]), z_start, z_step, n_samples).T
        assert np.array_equal(by_mol[j], want, equal_nan=True), (j, X[:, j], V[:, j])
        assert w1[j] == np.isfinite(want[:, 5]).sum() or not np.isfinite(np.r_[X[:, j], V[:, j]]).all()


@pytest.mark.parametrize("field", ["hexapole", "linear"])
@pytest.mark.parametrize("grid", [(0.0, 1e-3, 1200), (-0.1, 0.05, 64), (0.3, 0.05, 65), (0.55, 1.7e-4, 700),
                                  (0.499999, 1e-7, 130), (0.2, 0.01, 63), (2.0, 0.1, 80)], ids=str)
def test_grids(field, grid):
    eng = Engine(beamline(field, plates=True))
    X, V = molecules(700, 3)
    slow = np.abs(V[2]) < 2  # ten thousand and more lens rows: compared between the layouts only
    check(eng, X, V, *grid, np.flatnonzero(~slow)[:300])


@pytest.mark.parametrize("n", [1, 511, 512, 575, 577])
@pytest.mark.parametrize("n_samples", [63, 64, 600])
def test_counts(n, n_samples):
    js = np.unique(np.r_[0:min(n, 20), max(0, n - 66):n])
    check(Engine(beamline("hexapole")), *molecules(n, n, odd=False), 0.0, 1.2 / n_samples, n_samples, js)


@pytest.mark.parametrize("length,dt", [(0.1, 1.0), (1e-6, 1e-5), (0.1, 1e-6)])  # no full step; one; thousands
def test_steps(length, dt):
    check(Engine(beamline("hexapole", length, dt)), *molecules(520, 1, odd=False), 0.45, 1e-3, 300, np.arange(70))


def test_more_than_a_slice_in_two_states():
    """A slice holds 128 MiB of face rows: of a beamline of 60 elements, 13 632 molecules."""
    n = 13_700
    X, V = molecules(n, 9, odd=False)
    X[2] = 0.0
    lens = ElectrostaticLens("ES lens", 0.1, 0.02, d=2 * configs.LENS_R, V=25e3,
                             stark=[configs.stark_table(-1.0), configs.stark_table(1.0)], field="hexapole",
                             integrator="rk4", dt=configs.LENS_DT)
    bl = Beamline([CircularAperture("A", 0.05, 0.0, d=12e-3), lens] +
                  [CircularAperture("B", 0.13 + 1e-4 * k, 0.0, d=12e-3) for k in range(58)], 9.81)
    js = np.r_[0:5, 63:66, 13_630:13_634, n - 3:n]
    check(Engine(bl, n_states=2), X, V, 0.0, 2e-3, 70, js, state=(np.arange(n) % 2).astype(np.uint8))


@pytest.mark.parametrize("n,n_samples", [(16_384, 64), (16_385, 255), (16_385, 256), (32_769, 256)])
def test_sample_counts_that_change_the_form(n, n_samples):
    X, V = molecules(n, 4, odd=False)
    js = np.r_[0:3, 16_382:16_384, n - 2:n]
    check(Engine(beamline("hexapole", 0.02)), X, V, 0.4, 0.2 / n_samples, n_samples, js)
