"""Chunked host draws refuse what the distributions' own draws refuse, draw nothing for no chunks, and go through a
draw method that an instance was given."""
import numpy as np
import pytest

from trajectories.distributions import (CeNTREXPositionDistribution, CeNTREXVelocityDistribution,
                                        GaussianPositionDistribution, draw_chunks)

NAN = float("nan")
X = [GaussianPositionDistribution(), CeNTREXPositionDistribution()]


@pytest.mark.parametrize("bad", [NAN, -1.0])
@pytest.mark.parametrize("which", ["sigmax", "sigmay", "sigmaz"])
@pytest.mark.parametrize("xd", X, ids=["gaussian", "disc"])
def test_widths_of_the_velocity(xd, which, bad):
    vd = CeNTREXVelocityDistribution(**{which: bad})
    with pytest.raises(ValueError):
        vd.draw(5)
    with pytest.raises(ValueError):
        draw_chunks(xd, vd, 5, 3)


@pytest.mark.parametrize("bad", [NAN, -1.0])
@pytest.mark.parametrize("which", [0, 1])
def test_widths_of_the_position(which, bad):
    widths = [1e-3, 1e-3]
    widths[which] = bad
    xd = GaussianPositionDistribution(*widths)
    with pytest.raises(ValueError):
        xd.draw(5)
    with pytest.raises(ValueError):
        draw_chunks(xd, CeNTREXVelocityDistribution(), 5, 3)


@pytest.mark.parametrize("xd", X, ids=["gaussian", "disc"])
@pytest.mark.parametrize("chunks", [0, -1])
def test_no_chunks(xd, chunks):
    state = np.random.get_state()
    A, B = draw_chunks(xd, CeNTREXVelocityDistribution(), 5, chunks)
    assert A.shape == B.shape == (3, 0)
    assert all(np.array_equal(a, b) for a, b in zip(state, np.random.get_state()))


@pytest.mark.parametrize("xd", X, ids=["gaussian", "disc"])
def test_a_draw_method_of_the_instance(xd):
    vd = CeNTREXVelocityDistribution()
    vd.draw = lambda n: np.full((3, n), 7.0)
    assert np.array_equal(draw_chunks(xd, vd, 5, 3)[1], np.full((3, 15), 7.0))
    own = type(xd)()
    own.draw = lambda n: np.full((3, n), 8.0)
    assert np.array_equal(draw_chunks(own, CeNTREXVelocityDistribution(), 5, 3)[0], np.full((3, 15), 8.0))
