"""GPU: circular-aperture walks of molecules at and beyond the limits of the short arithmetic.

Molecules of moderate size walk with one shared reciprocal of vz and without the products that are zero; others
(vz or z outside [2^-100, 2^100) except z = 0, x or vx = -0, given accelerations) and beamlines with faces outside
that range walk plainly.  Both are the oracle's operations, so a mixture equals the oracle bit for bit, on beamlines
without a lens, before and after one, and in the batched scan.
"""
import numpy as np
import pytest

from oracle import oracle as O
from trajectories import _native as N
from trajectories import configs
from trajectories.batch import BatchScan
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture
from trajectories.engine import Engine

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "t")


def molecules(n, seed):
    rs = np.random.RandomState(seed)
    pick = lambda values: rs.choice(values, n)  # noqa: E731
    x = np.where(rs.rand(n) < 0.5, rs.normal(0, 2e-3, n), pick([0.0, -0.0, 2.0 ** -120, -1e-300, 5e-3, 6e-3]))
    y = np.where(rs.rand(n) < 0.5, rs.normal(0, 2e-3, n), pick([0.0, -0.0, 2.0 ** -120, 1e-310, -5e-3]))
    z = pick([0.0, -0.0, 0.1, 0.3, -0.2, 2.0 ** -99, 2.0 ** -101, 2.0 ** 101, np.nan])
    vx = np.where(rs.rand(n) < 0.7, rs.normal(0, 1.5, n), pick([0.0, -0.0, np.inf, 1e-200]))
    vy = np.where(rs.rand(n) < 0.7, rs.normal(0, 1.5, n), pick([0.0, -0.0, -np.inf, 1e-200]))
    vz = np.where(rs.rand(n) < 0.6, rs.normal(184.0, 16.0, n),
                  pick([184.0, -50.0, 2.0 ** -99, 2.0 ** -101, 2.0 ** 99, 2.0 ** 101, 0.0, -0.0, np.inf, np.nan]))
    return np.array([x, y, z]), np.array([vx, vy, vz])


def compare(bl, X, V, a0=None, t=None):
    eng = Engine(bl)
    with np.errstate(all="ignore"):
        o = O.propagate(eng.cb, *X, *V, t, a0=a0)
    for flags in (0, N.RUN_SIMPLE):
        d = eng.propagate(*X, *V, t, a0=a0, flags=flags, want_accel=True)
        assert np.array_equal(d["label"], o["label"])
        for k in FIELDS:
            assert np.array_equal(d["out"][k], o["out"][k], equal_nan=True), (flags, k)
            assert np.array_equal(np.signbit(d["out"][k]), np.signbit(o["out"][k])) or np.isnan(o["out"][k]).any(), k
        for q in range(3):
            assert np.array_equal(d["out_a"][q], o["out_a"][q], equal_nan=True)
        assert int(d["work"][N.WORK_FACES]) == int(o["work"][0])
    # runs without per-molecule outputs (two-deep prefetch)
    r = eng.propagate(*X, *V, t, a0=a0, outputs=False, per_molecule=False, aoi_labels=list(eng.labels))
    order = np.argsort(r["aoi_index"])
    assert np.array_equal(r["aoi_index"][order], np.arange(X.shape[1]))
    for k in FIELDS:
        assert np.array_equal(r["aoi_out"][k][order], o["out"][k], equal_nan=True), k


FACES = [[(0.3, 0.0), (0.8, 0.01), (1.2, 0.0)], [(0.0, 0.0), (0.5, 0.1)], [(2.0 ** -101, 0.1)], [(0.3, 2.0 ** 101)]]


@pytest.mark.parametrize("faces", FACES, ids=str)
@pytest.mark.parametrize("n", [1, 63, 5000])
def test_apertures(faces, n):
    bl = Beamline([CircularAperture(f"A{k}", z0, L, d=1e-2) for k, (z0, L) in enumerate(faces)], 9.81)
    X, V = molecules(n, n)
    compare(bl, X, V)
    rs = np.random.RandomState(n)
    compare(bl, X, V, a0=[rs.normal(0, 3.0, n), rs.normal(0, 3.0, n), rs.normal(0, 3.0, n)], t=rs.rand(n))


@pytest.mark.parametrize("g", [0.0, 9.81, -2.0, 2.0 ** -110])
def test_gravity(g):
    X, V = molecules(3000, 8)
    compare(Beamline([CircularAperture("A", 0.3, 0.0, d=1e-2), CircularAperture("B", 0.9, 0.2, d=1e-2)], g), X, V)


def test_around_a_lens():
    X, V = molecules(4000, 9)
    X[0, ::2], X[1, ::2] = X[0, ::2] * 0.3, X[1, ::2] * 0.3
    keep = np.isfinite(X).all(0) & np.isfinite(V).all(0) & (V[2] > 1.0) & (V[2] < 1e4)  # the step cap aside
    for bl in (configs.config1(stark=configs.stark_table(+1.0)), configs.config1(lens_z0=0.5)):
        compare(bl, X[:, keep], V[:, keep])


def test_batch_equals_single_runs():
    bls = [configs.config1(V0=2e4), configs.config1(V0=3e4, lens_z0=0.7), configs.config0()]
    n, seeds = [3000, 1, 5000], [5, 6, 7]
    sigma = np.array(configs.SOURCE_SIGMA) * [1, 1, 1, 1, 1, 8]  # some molecules with vz <= 0
    tally = BatchScan(bls, n, seeds, configs.SOURCE_MEAN, sigma).run()[0]
    scan_labels = BatchScan(bls, n, seeds, configs.SOURCE_MEAN, sigma).labels
    for c, bl in enumerate(bls):
        eng = Engine(bl)
        d = [a.to_host(count=n[c]) for a in eng.draw_gaussian(n[c], configs.SOURCE_MEAN, sigma, seeds[c])]
        r = O.propagate(eng.cb, *d)
        want = dict(zip(eng.labels, np.bincount(r["label"], minlength=len(eng.labels))))
        assert {k: v for k, v in zip(scan_labels, tally[c].tolist()) if v} == {k: v for k, v in want.items() if v}
