"""GPU: the signs of zeros through circular-aperture walks, molecule by molecule against the oracle.

A molecule that stands on a face is left as it is there (a drift of no time), so its zeros keep their signs: starts
on, before and behind the first face, beamlines that end there or go on, with every sign of x, y, vx, vy
and t, under gravity of either sign and none.
"""
import itertools

import numpy as np
import pytest

from oracle import oracle as O
from trajectories import _native as N
from trajectories import configs
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture
from trajectories.engine import Engine

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "t")


def molecules(zs, vzs):
    """Every combination of signs and zeros: X, V (3, n) and t (n)."""
    v = [0.0, -0.0, 1e-3, -1e-3]
    m = np.array(list(itertools.product(v, v, zs, v, v, vzs, [0.0, -0.0, 0.5]))).T
    return m[0:3].copy(), m[3:6].copy(), m[6].copy()


def same(got, want, what):
    assert np.array_equal(got, want, equal_nan=True), what
    differ = np.flatnonzero((np.signbit(got) != np.signbit(want)) & ~np.isnan(want))
    assert differ.size == 0, (what, differ[:5], got[differ[:5]], want[differ[:5]])


def check(bl, X, V, t):
    eng = Engine(bl)
    n = X.shape[1]
    with np.errstate(all="ignore"):
        o = O.propagate(eng.cb, *X, *V, t)
    for flags in (0, N.RUN_SIMPLE):
        d = eng.propagate(*X, *V, t, flags=flags)
        for k in FIELDS:
            same(d["out"][k], o["out"][k], (flags, k))
    r = eng.propagate(*X, *V, t, outputs=False, per_molecule=False, aoi_labels=list(eng.labels))
    order = np.argsort(r["aoi_index"])
    assert np.array_equal(r["aoi_index"][order], np.arange(n))
    for k in FIELDS:
        same(r["aoi_out"][k][order], o["out"][k], ("kept", k))


@pytest.mark.parametrize("g", [0.0, -0.0, 9.81, -2.0])
@pytest.mark.parametrize("with_t", [True, False])
@pytest.mark.parametrize("more", [[], [(0.25, 0.0)], [(0.5, 0.25)]], ids=str)
def test_apertures(g, with_t, more):
    faces = [(0.25, 0.0)] + more
    bl = Beamline([CircularAperture(f"A{k}", z0, L, d=1e-2) for k, (z0, L) in enumerate(faces)], g)
    X, V, t = molecules([0.0, -0.0, 0.25, 1.0], [2.0, -2.0])
    check(bl, X, V, t if with_t else None)


def test_before_a_lens():
    X, V, t = molecules([0.3, 0.1], [184.0])
    check(configs.config1(), X, V, t)
