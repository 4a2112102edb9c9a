"""GPU: the reference lens's step for states where its fast form does not apply, or applies at its limits.

The fast form (shared reciprocals, no scaling for extreme exponents) holds while the state lies in
[2^-200, 2^200) and every force evaluation in the guessed table segment; other lanes take the plain step.  Both
are the oracle's operations bit for bit, so a mixture of them is compared with the oracle exactly: axis
molecules (zero coordinates), coordinates around 2^-200 and far below it, velocities that leave the table or
reach 2^200 and infinity, radii at and next to the table's knots, and tables that are not of moderate size.
"""
import numpy as np
import pytest

from oracle import oracle as O
from trajectories import _native as N
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens
from trajectories.beamline_elements.electrostatic_lens import LinearTable
from trajectories.engine import Engine
from trajectories.stark import TwoLevelStark

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "t")


def beamline(table=None, L=0.05, dz=1e-3):
    lens = ElectrostaticLens("ES lens", 0.1, L, dz=dz, a_interp=table, state=TwoLevelStark(sign=1.0))
    return Beamline([lens, CircularAperture("end", 0.3, 0.0, d=0.02)])


def compare(bl, X, V):
    eng = Engine(bl)
    with np.errstate(all="ignore"):
        o = O.propagate(eng.cb, *X, *V)
    for flags in (0, N.RUN_LANES, N.RUN_SIMPLE):
        d = eng.propagate(*X, *V, flags=flags)
        assert np.array_equal(d["label"], o["label"]) and np.array_equal(d["status"], o["status"])
        for k in FIELDS:
            assert np.array_equal(d["out"][k], o["out"][k], equal_nan=True), (flags, k)


def test_extreme_states():
    tiny = [0.0, -0.0, 2.0 ** -199, 2.0 ** -200, 2.0 ** -201, 2.0 ** -400, 2.0 ** -1060, 1e-9, 1e-4, 3e-3]
    fast = tiny + [1.0, 40.0, 1e3, 2.0 ** 199, 2.0 ** 200, 2.0 ** 600, np.inf, np.nan]
    rs = np.random.RandomState(3)
    n = 4000
    pick = lambda values: rs.choice(values, n) * rs.choice([1.0, -1.0], n)  # noqa: E731
    X = np.vstack([pick(tiny), pick(tiny), np.zeros(n)])
    V = np.vstack([pick(fast), pick(fast), rs.choice([184.0, 150.0, 2.0 ** -190, 2.0 ** 198, 2.0 ** 205], n)])
    compare(beamline(), X, V)


def test_knots():
    """Molecules that enter the lens on a knot, one ulp beside it and at the table's end."""
    r = np.linspace(0, 1.75 * 0.0254 / 2 * 1.01, 222)
    near = np.concatenate([r, np.nextafter(r, -1.0), np.nextafter(r, 1.0)])
    X = np.vstack([near, np.zeros_like(near), np.full_like(near, 0.1)])
    V = np.vstack([np.zeros_like(near), np.zeros_like(near), np.full_like(near, 184.0)])
    X[1, 1::2] = 1e-30
    compare(beamline(LinearTable(r, -3e4 * np.sin(r * 300.0))), X, V)


@pytest.mark.parametrize("scale", [0.0, 2.0 ** -210, 1.0, 2.0 ** 210])
@pytest.mark.parametrize("n", [1, 64, 1000])
def test_tables(scale, n):
    r = np.concatenate([np.linspace(0.0, 0.01, 50), np.linspace(0.011, 0.024, 30)])  # two spacings: guesses miss
    rs = np.random.RandomState(n)
    X = np.vstack([rs.normal(0, 3e-3, (2, n)), np.zeros(n)])
    V = np.vstack([rs.normal(0, 2.0, (2, n)), rs.normal(184.0, 16.0, n)])
    compare(beamline(LinearTable(r, scale * -2e4 * r / 0.02)), X, V)
