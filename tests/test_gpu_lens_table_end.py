"""GPU: lens steps with and without the clamp to the force table's end.

Wavefronts whose molecules provably stay inside the table step without the clamp.  The table's end is
set as a multiple of the field at the bore: inside the bore (every molecule may clamp), just beyond it
(the bound allows none), where it allows some of them, and where it allows all; the molecules include
ones that are far too fast and ones that are not finite.  Bits of the one-molecule-per-thread walker,
which always clamps; the scan's tallies are those of its single-kernel walker, which always clamps too.
"""
import numpy as np
import pytest

from trajectories import _native as N
from trajectories import configs
from trajectories._native import BatchTune
from trajectories.batch import BatchScan
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens
from trajectories.engine import Engine
from trajectories.stark import TwoLevelStark, WSpline

pytestmark = pytest.mark.gpu

V, LENGTH, KNOTS = 25e3, 0.3, 1001
BORE_FIELD = 4.29e4  # V/cm at the bore of this lens


def tables_to(factor, states=1):
    return [WSpline.from_stark(TwoLevelStark(configs.NU, configs.MU_D, s, d), BORE_FIELD * factor, KNOTS)
            for s, d in ((-1.0, 1.0), (1.0, 0.7))][:states]


def beamline(tables, V=V):
    states = len(tables)
    lens = ElectrostaticLens("ES lens", 0.8, LENGTH, d=2 * configs.LENS_R, V=V,
                             stark=tables if states > 1 else tables[0],
                             field="hexapole", integrator="rk4", dt=configs.LENS_DT)
    return Beamline([CircularAperture("A", 0.3, 0.0, d=2 * configs.LENS_R), lens,
                     CircularAperture("B", 1.6, 0.0, d=6e-3)], 9.81)


def molecules(n, seed):
    rs = np.random.RandomState(seed)
    X = np.vstack([rs.normal(0, configs.SIGMA_X, (2, n)), np.zeros(n)])
    U = np.vstack([rs.normal(0, configs.SIGMA_V, (2, n)), rs.normal(configs.VZ_MEAN, configs.VZ_SIGMA, n)])
    odd = rs.permutation(n)[: n // 50]
    U[0, odd] = rs.choice([1e3, -1e4, 1e300, np.inf, np.nan], odd.size)
    # fast ones that reach the lens: they pass the entrance at its axis
    k = odd[: odd.size // 2]
    U[0, k] = rs.choice([300.0, -2e3, 5e4], k.size)
    X[0, k] = -U[0, k] / U[2, k] * 0.8
    return X, U


FACTORS = [0.5, 0.999, 1.001, 1.03, 1.06, 2.4]


@pytest.mark.parametrize("states", [1, 2])
@pytest.mark.parametrize("factor", FACTORS)
def test_same_bits_as_with_the_clamp(factor, states):
    eng = Engine(beamline(tables_to(factor, states)))
    for n in (777, 150_001):  # queue regions; claim list
        X, U = molecules(n, n)
        kw = dict(state=(np.arange(n) % 2).astype(np.uint8)) if states > 1 else {}
        ref = eng.propagate(*X, *U, flags=N.RUN_SIMPLE, **kw)
        got = eng.propagate(*X, *U, **kw)
        for k in ("tally", "first_index", "label", "status"):
            assert np.array_equal(got[k], ref[k]), k
        assert np.array_equal(got["work"][:4], ref["work"][:4])
        for k, v in ref["out"].items():
            assert np.array_equal(got["out"][k], v, equal_nan=True), k


@pytest.mark.parametrize("factor", FACTORS)
def test_scan_tallies(ctx, factor):
    tables = tables_to(factor)
    bls = [beamline(tables), beamline(tables, 0.9 * V)]  # the bound is the smaller of the two lenses'
    counts, seeds = np.array([5000, 77]), np.array([1, 2], dtype=np.uint64)
    sigma = np.array(configs.SOURCE_SIGMA, float) * [1, 1, 1, 3, 3, 1]
    scan = BatchScan(bls, counts, seeds, configs.SOURCE_MEAN, sigma, ctx=ctx)
    tally, work, _ = scan.run(BatchTune(block=0, chunk=128, grid=0, refill=0, use_graph=0, fused=0))
    fused, fwork, _ = scan.run(BatchTune(block=0, chunk=128, grid=0, refill=0, use_graph=0, fused=1))
    np.testing.assert_array_equal(tally, fused)
    np.testing.assert_array_equal(work[:4], fwork[:4])
