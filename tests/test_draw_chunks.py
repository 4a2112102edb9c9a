"""Chunked host draws equal scipy's calls in the reference's order, value for value and in the state they leave."""
import numpy as np
import pytest
from scipy.stats import norm, uniform

from trajectories.distributions import (CeNTREXPositionDistribution, CeNTREXVelocityDistribution, GaussianDistribution,
                                        GaussianPositionDistribution, draw_chunks)


def normal(loc, scale, n):
    return norm.rvs(loc=loc, scale=scale, size=n)


def reference_draws(xd, vd, n, chunks):
    """run_simulation's draws (trajectory_simulator.py:52-60) with scipy's own calls."""
    xs, vs = [], []
    for _ in range(chunks):
        vs.append(np.array([normal(vd.vx, vd.sigmax, n), normal(vd.vy, vd.sigmay, n), normal(vd.vz, vd.sigmaz, n)]))
        if isinstance(xd, GaussianPositionDistribution):
            xs.append(np.vstack([normal(0, xd.sigmax, n), normal(0, xd.sigmay, n), np.full(n, xd.z)]))
        else:
            theta = uniform.rvs(size=n) * 2 * np.pi
            r = np.sqrt(uniform.rvs(size=n)) * xd.d / 2
            xs.append(np.array([r * np.cos(theta), r * np.sin(theta), np.full(n, xd.z)]))
    return np.concatenate(xs, axis=1), np.concatenate(vs, axis=1)


@pytest.mark.parametrize("n,chunks", [(1, 1), (1, 100), (7, 33), (10, 100), (1001, 10)])
@pytest.mark.parametrize("xd", [CeNTREXPositionDistribution(), CeNTREXPositionDistribution(d=1, z=0),
                                GaussianPositionDistribution(1.5e-3, 2e-3, 0.0), GaussianPositionDistribution(0.0, 1.0)],
                         ids=str)
@pytest.mark.parametrize("vd", [CeNTREXVelocityDistribution(), CeNTREXVelocityDistribution(0, 1.5, 0, 1.5, 184, 16),
                                CeNTREXVelocityDistribution(sigmay=0.0)], ids=str)
def test_chunks_replay_scipy(xd, vd, n, chunks):
    states, draws = [], []
    for f in (reference_draws, draw_chunks):
        np.random.seed(4)
        np.random.standard_normal(1)  # a cached second normal
        draws.append(f(xd, vd, n, chunks))
        states.append(np.random.get_state())
    for a, b in zip(*draws):
        assert a.dtype == b.dtype == np.float64 and np.array_equal(a, b)
    assert all(np.array_equal(a, b) for a, b in zip(*states))


def test_other_distributions_and_arguments():
    class Doubled(CeNTREXVelocityDistribution):
        def draw(self, n):
            return 2.0 * super().draw(n)

    np.random.seed(1)
    _, V = draw_chunks(GaussianPositionDistribution(), Doubled(), 5, 4)
    np.random.seed(1)
    _, W = draw_chunks(GaussianPositionDistribution(), CeNTREXVelocityDistribution(), 5, 4)
    assert np.array_equal(V, 2.0 * W)
    assert draw_chunks(GaussianPositionDistribution(), CeNTREXVelocityDistribution(), 0, 100)[0].shape == (3, 0)
    with pytest.raises(ValueError):
        GaussianDistribution(0.0, -1.0).draw(3)
    np.random.seed(2)
    a = GaussianDistribution(np.array([1.0, 2.0]), 3.0).draw(2)
    np.random.seed(2)
    assert np.array_equal(a, normal(np.array([1.0, 2.0]), 3.0, 2))
