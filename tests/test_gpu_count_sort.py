"""GPU: the counting sort at the cell sizes where it reads the members in other batches (8,
then 16 at a time) and at the edge counts around a batch of 4, against the tile sort: the
same order, so the same state, counts and graphs bit for bit; one simulation and several."""

import numpy as np
import pytest

from cellflow_amd import Ensemble
from helpers import make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 16, 17, 23, 24, 25, 40, 41, 300]


def clumped(extra):
    """A clump of each size, every clump within a cell of its own (0.1 apart), and singles."""
    cfg = small_cfg(n=sum(SIZES) + extra, side=0.8, T=2, seed=extra + 1)
    st, phys, params = state_of(cfg)
    rng = np.random.default_rng(extra)
    sites = np.stack(np.meshgrid(*[np.arange(0.05, 0.8, 0.1)] * 3), -1).reshape(-1, 3)
    sites = sites[rng.permutation(len(sites))[: len(SIZES)]]
    at = np.repeat(sites, SIZES, axis=0) + rng.uniform(-0.003, 0.003, (sum(SIZES), 3))
    order = rng.permutation(cfg["n"])[: sum(SIZES)]
    st["pos"][order] = at.astype(np.float32)
    return st, phys, params


@pytest.mark.parametrize("extra", [0, 63, 1000])
@pytest.mark.parametrize("maxc", [3, 8, 32])
def test_counting_sort_equals_tile_sort(extra, maxc):
    st, phys, params = clumped(extra)
    out = []
    for sort in (0, 1):
        sim = make_sim(st, phys)
        sim.setTuning(sort_variant=sort)
        sim.simulate(params, 3, edges=(0.01, maxc))
        out.append((sim.getParticleData().tobytes(), sim.getNeighborCounts().tobytes(),
                    sim.getEdges().tobytes(), sim.getStepEdges().tobytes()))
        assert len(sim.getStepEdges()) > 0
        sim.close()
    assert out[0] == out[1]


def test_counting_sort_of_an_ensemble():
    sims = [(clumped(e)[1], clumped(e)[0]) for e in (0, 63, 130)]
    out = []
    for sort in (0, 1):
        ens = Ensemble(sims)
        ens.setTuning(sort_variant=sort)
        ens.simulate(3)
        out.append([ens.getParticleData(s).tobytes() for s in range(3)])
        ens.close()
    assert out[0] == out[1]
