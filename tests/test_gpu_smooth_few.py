"""GPU: gradients of few molecules, whose work items are spread over the CUs.

The sums are added item by item in a fixed order, so the workgroup's size changes no bit; and the library's choice is
no slower than the workgroups of eight wavefronts that it took before it kept sixteen on a CU.
"""
import time

import numpy as np
import pytest

from trajectories import configs
from trajectories.smooth import SmoothFlux

pytestmark = pytest.mark.gpu


def flux(n, block=0):
    src = [a[:n] for a in configs.config3_source((n + 99) // 100 * 100, 7)]
    return SmoothFlux(configs.config1(stark=configs.stark_table(+1.0)), *src, sigma_vz=configs.VZ_SIGMA,
                      softness=configs.CONFIG3_SOFTNESS, block=block)


def sets(k):
    P = np.tile(configs.config3_theta(), (k, 1))
    P[:, 1] *= np.linspace(1.0, 1.1, k)
    return P


# one item; one for each CU, one more, and one fewer and more than two; many sets of one item; sixteen on each
@pytest.mark.parametrize("n,k", [(1, 1), (64 * 256, 1), (64 * 256 + 1, 1), (64 * 512 - 64, 1), (64 * 512 + 1, 1),
                                 (40, 300), (64 * 256 * 16 + 1, 1)])
def test_the_choice_changes_no_bit(n, k):
    want = None
    for block in (0, 64, 256, 512):
        r = flux(n, block).evaluate(sets(k))
        if want is None:
            want = r
        assert np.array_equal(r.J, want.J) and np.array_equal(r.grad, want.grad)


@pytest.mark.parametrize("n", [1000, 16_384, 65_536, 131_072])
def test_the_choice_is_not_slower(n):
    def us(pr):
        P, best = configs.config3_theta(), np.inf
        for _ in range(12):
            a = time.perf_counter()
            pr.evaluate(P)
            best = min(best, time.perf_counter() - a)
        return best * 1e6

    own, eight = us(flux(n)), us(flux(n, 512))
    assert own <= 1.15 * eight, (own, eight)
