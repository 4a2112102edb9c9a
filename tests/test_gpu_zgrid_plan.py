"""GPU: z-grid samples where the number of lens steps decides their form.

Rows that outgrow the workspace in the middle of a slice (molecules that an axial acceleration slows down before the
lens, which the plan made from vz cannot know), step counts on both sides of the room and of the bounds of the rule, one
molecule that moves backwards among many, and several slices: every sample is that of the oracle's sampling of the
molecule's own recorded rows, in both layouts.  And a call takes no longer than the walk of a few molecules by the
one-kernel form, whose serial steps bound it.
"""
import ctypes as C
import time

import numpy as np
import pytest

from oracle import oracle as O
from trajectories import _native as N
from trajectories import configs
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens
from trajectories.engine import Engine, bind

pytestmark = pytest.mark.gpu


def engine(length, dt):
    lens = ElectrostaticLens("ES lens", 0.3, length, d=2 * configs.LENS_R, V=25e3, stark=configs.stark_table(),
                             field="hexapole", integrator="rk4", dt=dt)
    return Engine(Beamline([CircularAperture("A", 0.2, 0.0, d=12e-3), lens,
                            CircularAperture("B", 1.0, 0.0, d=6e-3)], 9.81))


def molecules(n, seed):
    rs = np.random.RandomState(seed)
    X = np.vstack([rs.normal(0, configs.SIGMA_X / 2, (2, n)), np.zeros(n)])
    V = np.vstack([rs.normal(0, configs.SIGMA_V / 4, (2, n)), rs.normal(configs.VZ_MEAN, configs.VZ_SIGMA, n)])
    return X, V


def check(eng, X, V, z_start, z_step, n_samples, js, a0=None):
    kw = dict(z_start=z_start, z_step=z_step, n_samples=n_samples, a0=a0)
    field, w1, l1 = eng.zgrid(*X, *V, **kw)
    by_mol, w2, l2 = eng.zgrid_by_molecule(*X, *V, **kw)
    assert np.array_equal(w1, w2) and np.array_equal(l1, l2)
    assert np.array_equal(field.transpose(2, 1, 0), by_mol, equal_nan=True)
    sub = None if a0 is None else [a[js] for a in a0]
    rows, n_rows, lab = eng.record_rows(*X[:, js], *V[:, js], a0=sub, cap=9000)
    assert np.array_equal(lab, l1[js]) and n_rows.max() <= 9000
    for q, j in enumerate(js):
        want = O.zgrid_from_rows(rows[q], int(n_rows[q]), z_start, z_step, n_samples).T
        assert np.array_equal(by_mol[j], want, equal_nan=True), (j, X[:, j], V[:, j])
        assert w1[j] == np.isfinite(want[:, 5]).sum()
    return n_rows


def test_rows_that_outgrow_the_workspace():
    """4096 molecules have room for 4.2e6 rows; the plan counts some 330 each, two thirds take 5000."""
    n = 4096
    X, V = molecules(n, 2)
    az = np.zeros(n)
    slow = np.random.RandomState(3).permutation(n)[: n // 3 * 2]
    az[slow] = -(V[2, slow] - 12.0) * V[2, slow] / 0.2  # 12 m/s once it has drifted for its time to the first element
    V[:2, slow] *= 0.02
    js = np.unique(np.r_[slow[:12], 0:12, n - 12:n])
    n_rows = check(engine(0.2, 3.3e-6), X, V, 0.0, 5e-3, 240, js, a0=[np.zeros(n), np.full(n, -9.81), az])
    assert (n_rows > 600).sum() >= 8  # slowed ones that came into the lens, where each asks for 5000 rows


@pytest.mark.parametrize("steps", [2, 30, 40, 300, 400, 1000, 1100])
@pytest.mark.parametrize("n,n_samples", [(600, 70), (16_384, 64), (40_960, 256), (33_000, 300)])
def test_steps_around_the_bounds(n, n_samples, steps):
    length = 0.02 if steps < 50 else 0.2
    X, V = molecules(n, steps)
    js = np.unique(np.r_[0:4, n // 2, n - 4:n])
    check(engine(length, length / (configs.VZ_MEAN * steps)), X, V, 0.1, 1.0 / n_samples, n_samples, js)


@pytest.mark.parametrize("vz", [-100.0, 0.0])
def test_one_molecule_that_does_not_move_forward(vz):
    n = 41_000  # in the second slice
    X, V = molecules(n, 5)
    V[2, n - 3] = vz
    js = np.r_[0:3, 40_958:40_962, n - 2:n]
    check(engine(0.1, 1e-5), X, V, 0.1, 1e-3, 260, js)


def us(eng, mode, n, n_samples):
    """The device time of one call, kept buffers and all."""
    X, V = molecules(n, 7)
    ctx = eng.ctx
    cols = [ctx.to_device(a) for a in (*X, *V)]
    buf = ctx.alloc(6 * n_samples * n)
    R = N.Record()
    R.n, R.mode, R.cap, R.z_start, R.z_step, R.buf = n, mode, n_samples, 0.0, 1.2 / n_samples, buf.ptr
    for name, col in zip(("x", "y", "z", "vx", "vy", "vz"), cols):
        setattr(R.inp, name, col.ptr)
    bind(ctx, eng.cb)
    best = np.inf
    for _ in range(12):
        ctx.sync()
        a = time.perf_counter()
        N.check("ctraj_record_trajectories", N.lib().ctraj_record_trajectories(ctx.handle, C.byref(R)), ctx.handle)
        ctx.sync()
        best = min(best, time.perf_counter() - a)
    return best * 1e6


MOL, FIELD = N.REC_ZGRID_MOL, N.REC_ZGRID


@pytest.mark.parametrize("mode,n,n_samples,dt,most", [
    (MOL, 600, 64, 5e-6, 1.2), (FIELD, 600, 64, 5e-6, 1.2), (MOL, 16_384, 64, 2e-6, 1.3), (FIELD, 16_384, 64, 2e-6, 1.3),
    (MOL, 37_000, 256, 5e-6, 1.5), (FIELD, 37_000, 256, 5e-6, 1.9)])
def test_more_steps_take_no_form_twice(mode, n, n_samples, dt, most):
    """With the workspace outgrown, walking some of the molecules by each form took 1.3 to 1.7 times as long as the
    one-kernel form for all, which takes 1 to 1.6 times as long for these as for 500 molecules."""
    eng = engine(0.6, dt)
    few, all_of_them = us(eng, mode, 500, n_samples), us(eng, mode, n, n_samples)
    assert all_of_them <= most * few, (all_of_them, few)


def test_few_steps_and_samples_take_the_one_kernel_form():
    eng = engine(0.02, 1e-5)
    assert us(eng, N.REC_ZGRID_MOL, 16_384, 64) <= 1.4 * us(eng, N.REC_ZGRID_MOL, 500, 64)
