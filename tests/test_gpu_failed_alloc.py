"""GPU: an allocation that fails is reported once, by its own call."""
import numpy as np
import pytest

from trajectories import _native as N
from trajectories import configs
from trajectories.device import Context
from trajectories.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["alloc", "scratch", "result"])
def test_the_next_call_does_not_see_it(kind):
    ctx = Context(0)
    eng = Engine(configs.config0(), ctx)
    X, V = configs.draw_source(1000, 3)
    want = eng.propagate(*X, *V)["label"]
    with pytest.raises(N.NativeError, match="memory"):
        getattr(ctx, kind)(1 << 47)
    assert np.array_equal(eng.propagate(*X, *V)["label"], want)
    ctx.close()
