"""GPU: buffers that a device-drawn run hands to a distribution."""
import numpy as np
import pytest

from trajectories import configs
from trajectories.device import ScratchArray
from trajectories.distributions import CeNTREXVelocityDistribution, GaussianPositionDistribution
from trajectories.trajectory_simulator import simulate_device

pytestmark = pytest.mark.gpu


class OwnPositions(GaussianPositionDistribution):
    seen = ()

    def draw_device(self, n, seed, offset=0, ctx=None, out=None):
        self.seen = list(out)
        return super().draw_device(n, seed, offset=offset, ctx=ctx, out=out)


def test_an_override_gets_memory_of_its_own():
    """It may fill them on any stream, so they are no blocks that the context's stream may still use."""
    x, v = (1.5e-3, 1.5e-3, 0.0), CeNTREXVelocityDistribution(0, 1.5, 0, 1.5, 184, 16)
    own = OwnPositions(*x)
    a = simulate_device(configs.config1(), own, v, 5000, 3, ["Detected"])
    b = simulate_device(configs.config1(), GaussianPositionDistribution(*x), v, 5000, 3, ["Detected"])
    assert len(own.seen) == 3 and not any(isinstance(o, ScratchArray) for o in own.seen)
    assert np.array_equal(a.tally, b.tally) and np.array_equal(a.aoi_index, b.aoi_index)
