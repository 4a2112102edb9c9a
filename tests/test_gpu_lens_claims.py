"""GPU: how the lens kernel's wavefronts claim the queue, at the edges of its rules.

Few molecules (64 per SIMD) are claimed as queue regions, one each; more go through a claim list, longest-lived
first (hexapole) or in queue order; chunks beyond the wavefronts' first come from counters.  Every way gives
the bits of the one-molecule-per-thread walker: final states, labels, tallies, first indices, step counts and
kept molecules.
"""
import numpy as np
import pytest

from trajectories import _native as N
from trajectories import configs
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens
from trajectories.engine import Engine
from trajectories.stark import TwoLevelStark

pytestmark = pytest.mark.gpu

EDGE = 64 * 4 * 256  # molecules up to which every SIMD of the device gets at most one region


def lens(kind):
    if kind == "reference":
        return ElectrostaticLens("ES lens", 0.8, 0.05, V=20e3, state=TwoLevelStark(sign=1.0))
    return ElectrostaticLens("ES lens", 0.8, 0.3, d=2 * configs.LENS_R, V=25e3, stark=configs.stark_table(),
                             field="hexapole", integrator="rk4", dt=configs.LENS_DT)


def beamline(kind, first):
    return Beamline([CircularAperture("A", 0.3, 0.0, d=2 * first), lens(kind),
                     CircularAperture("B", 1.6, 0.0, d=2 * 3e-3)], 9.81)


def molecules(n, seed):
    rs = np.random.RandomState(seed)
    X = np.vstack([rs.normal(0, configs.SIGMA_X, (2, n)), np.zeros(n)])
    V = np.vstack([rs.normal(0, configs.SIGMA_V, (2, n)), rs.normal(configs.VZ_MEAN, configs.VZ_SIGMA, n)])
    return X, V


def check(eng, X, V, **kw):
    ref = eng.propagate(*X, *V, flags=N.RUN_SIMPLE, aoi_labels=["B", "Detected"])
    for outputs in (True, False):
        got = eng.propagate(*X, *V, outputs=outputs, per_molecule=outputs, aoi_labels=["B", "Detected"], **kw)
        for k in ("tally", "first_index"):
            assert np.array_equal(got[k], ref[k]), (k, outputs)
        assert np.array_equal(got["work"][:4], ref["work"][:4])
        if outputs:
            assert np.array_equal(got["label"], ref["label"]) and np.array_equal(got["status"], ref["status"])
            for k, v in ref["out"].items():
                assert np.array_equal(got["out"][k], v, equal_nan=True), k
        o, p = np.argsort(got["aoi_index"]), np.argsort(ref["aoi_index"])
        assert np.array_equal(got["aoi_index"][o], ref["aoi_index"][p])
        for k, v in ref["aoi_out"].items():
            assert np.array_equal(got["aoi_out"][k][o], v[p]), k


@pytest.mark.parametrize("kind", ["hexapole", "reference"])
@pytest.mark.parametrize("n", [1, 63, 65, EDGE - 1, EDGE, EDGE + 1])
def test_counts(kind, n):
    eng = Engine(beamline(kind, 6e-3))
    check(eng, *molecules(n, n))


@pytest.mark.parametrize("kind", ["hexapole", "reference"])
@pytest.mark.parametrize("first", [1e-6, 1e-4, 1e-3])  # no, few or some molecules reach the lens
def test_sparse_queue(kind, first):
    check(Engine(beamline(kind, first)), *molecules(200_003, 5))


@pytest.mark.parametrize("kind", ["hexapole", "reference"])
@pytest.mark.parametrize("kw", [dict(flags=N.RUN_QUEUE_ORDER), dict(noalloc=True), dict(refill=1), dict(refill=64),
                                dict(block=64), dict(block=1024)], ids=str)
def test_ways_of_claiming(kind, kw):
    eng = Engine(beamline(kind, 6e-3))
    for n in (5000, 700_001):  # direct; more chunks than wavefronts
        check(eng, *molecules(n, 11), **kw)
