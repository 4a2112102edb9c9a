"""GPU: the smoothed flux at the edges of its work items, checkpoint windows and stores.

The reverse sweep recomputes the lens in windows of four steps from checkpoints taken every four steps, or
at the caller's interval where that store would grow too large (a huge max_steps forces it here).  Gradients
are compared with the CPU adjoint at the tolerance of the other adjoint tests (1e-10: sums of up to 10^3
molecules in another order, some 10^3 roundings of 1e-16 each along a trajectory), and with each other bit for
bit, since every store recomputes the same states.
"""
import numpy as np
import pytest

from oracle import oracle as O
from trajectories import configs
from trajectories.beamline import Beamline
from trajectories.beamline_elements import CircularAperture, ElectrostaticLens
from trajectories.smooth import SmoothFlux

pytestmark = pytest.mark.gpu


def source(n):
    return [a[:n] for a in configs.config3_source(1100, 7)]


def beamline(L):
    lens = ElectrostaticLens("ES lens", 0.8, L, d=2 * configs.LENS_R, V=30e3, stark=configs.stark_table(+1.0),
                             field="hexapole", integrator="rk4", dt=configs.LENS_DT)
    return Beamline([CircularAperture("A", 0.3, 0.01, d=12e-3), lens, CircularAperture("B", 1.6, 0.0, d=6e-3)], 9.81)


def compare(bl, src, theta, **kw):
    pr = SmoothFlux(bl, *src, sigma_vz=configs.VZ_SIGMA, softness=configs.CONFIG3_SOFTNESS, **kw)
    r = pr.evaluate(theta)
    o = O.smooth(pr.engine.cb, *src, theta, sigma_vz=configs.VZ_SIGMA, softness=configs.CONFIG3_SOFTNESS,
                 max_steps=pr.steps_needed(theta))
    assert r.J[0] == pytest.approx(o["J"][0], rel=1e-12, abs=1e-300)
    g, ref = r.grad[0] * theta, o["grad"][0] * theta
    assert np.all(np.abs(g - ref) <= 1e-10 * np.maximum(np.abs(ref), 1e-2 * np.abs(ref).max())), (g, ref)
    return r


THETA = np.array([6e-3, 30e3, 0.8, 3e-3, configs.VZ_MEAN])


# L: less than one step (partial step only), one to a few windows, windows and a remainder, the workload's
@pytest.mark.parametrize("L", [1e-3, 6e-3, 9e-3, 31e-3, 0.6])
@pytest.mark.parametrize("n", [1, 64, 65, 1000])
def test_window_edges(L, n):
    compare(beamline(L), source(n), THETA)


@pytest.mark.parametrize("every", [1, 3, 4, 5, 8, 64])
def test_stores_agree(every):
    bl, src = beamline(0.6), source(300)
    a = compare(bl, src, THETA, ckpt_every=8)
    for max_steps in (None, 1 << 18) if every > 4 else (None,):  # 2^18: too many for a checkpoint every four steps
        b = SmoothFlux(bl, *src, sigma_vz=configs.VZ_SIGMA, softness=configs.CONFIG3_SOFTNESS, ckpt_every=every,
                       max_steps=max_steps).evaluate(THETA)
        assert np.array_equal(a.J, b.J) and np.array_equal(a.grad, b.grad)


def test_unfolded_field_scale_takes_the_plain_step():
    compare(beamline(31e-3), source(200), THETA * [1, 1e-190, 1, 1, 1])
