"""Calls that fail leave the simulation as it was."""

import numpy as np
import pytest

from cellflow_amd import CellFlowError
from helpers import make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sort_variant", [0, 1])
@pytest.mark.parametrize("n", [100, 3000])
def test_failed_seeded_init_keeps_the_state(n, sort_variant):
    """A seeded init at a radius that is not finite is refused, and the particles stay."""
    st, phys, params = state_of(small_cfg(n=n))
    side = phys["canvas"][0]
    with make_sim(st, phys) as sim:
        sim.setTuning(sort_variant=sort_variant)
        sim.simulate(params, 7)
        before, counts = sim.getParticleData(), sim.getNeighborCounts()
        good = sim.getRadioByType()
        bad = good.copy()
        bad[1] = np.inf
        sim.setRadioByType(bad)
        with pytest.raises(CellFlowError, match="not finite"):
            sim.initializeParticles(3, phys["canvas"], side)
        sim.setRadioByType(good)
        assert sim.getParticleData().tobytes() == before.tobytes()
        assert np.array_equal(sim.getNeighborCounts(), counts)
        # and goes on as one that saw no failed call
        sim.simulate(params, 3)
        got = sim.getParticleData()
        sim.initializeParticles(3, phys["canvas"], side)
        fresh = sim.getParticleData()
    with make_sim(st, phys) as twin:
        twin.setTuning(sort_variant=sort_variant)
        twin.simulate(params, 7)
        twin.simulate(params, 3)
        assert twin.getParticleData().tobytes() == got.tobytes()
        twin.initializeParticles(3, phys["canvas"], side)
        assert twin.getParticleData().tobytes() == fresh.tobytes()
