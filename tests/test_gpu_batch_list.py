"""GPU: the scan's list of molecules that leave their lens, kept 64 entries at a time per wavefront.

A long lens that no molecule is stopped in sends every one of them through the list, a narrow one
hardly any; the counts stand around the 64 entries of a reservation.  Thresholds of 1 and 64 idle
lanes list one molecule and a whole wavefront at a time.  Tallies are whole numbers and equal those
of per-configuration propagation, which does not use the list, whatever the workgroup and grid.
"""
import numpy as np
import pytest

from trajectories import configs
from trajectories._native import BatchTune
from trajectories.batch import BatchScan
from trajectories.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma_scale", [0.02, 1.0])  # nearly all leave the lens; nearly all stop before or in it
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 129, 4097])
def test_listed_molecules_tally_as_per_configuration(ctx, n, sigma_scale):
    bls = [configs.config1(V0=30e3), configs.config1(V0=12e3, lens_z0=0.72)]
    counts = np.array([n, 2 * n + 1])
    seeds = np.array([7, 8], dtype=np.uint64)
    mean = np.array(configs.SOURCE_MEAN, float)
    sigma = np.array(configs.SOURCE_SIGMA, float) * sigma_scale
    scan = BatchScan(bls, counts, seeds, mean, sigma, ctx=ctx)
    want = []
    for c, bl in enumerate(bls):
        eng = Engine(bl, ctx)
        x = [a.to_host() for a in eng.draw_gaussian(int(counts[c]), mean, sigma, int(seeds[c]))]
        t = eng.propagate(*x, outputs=False)["tally"].sum(axis=0)
        want.append({k: int(v) for k, v in zip(eng.labels, t) if v})
    for block, grid, refill in ((0, 0, 0), (64, 1, 1), (64, 1, 64), (1024, 2, 8), (768, 0, 63)):
        tally, _, _ = scan.run(BatchTune(block=block, chunk=128, grid=grid, refill=refill, use_graph=0, fused=0))
        for c in range(2):
            got = {scan.labels[k]: int(tally[c, k]) for k in range(len(scan.labels)) if tally[c, k]}
            assert got == want[c], (block, grid, refill, c)
