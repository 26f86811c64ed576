"""GPU: the default tuning's force kernel (variant 0 at 16 lanes) at 8 and at 16 lanes per
particle, its list and its walk, and the wave's edge selection.

The kernel takes 16 lanes below 28,672 slots of the engine and 8 above, with the same order
of summation, so a member of a large ensemble (8 lanes) must equal its stand-alone run (16
lanes) bit for bit.  Graphs are compared with the oracle's, bit for bit.
"""

import numpy as np
import pytest

from cellflow_amd import Ensemble, SimulationParams
from helpers import check_step_edges, make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu

# (particles, box side, blobs, blob sd): list only; several list passes; walk; small grids
MEMBERS = [(1, 0.5, 0, 0), (64, 0.3, 0, 0), (65, 0.1, 0, 0), (2999, 0.6, 0, 0),
           (4097, 0.5, 0, 0), (5003, 0.9, 6, 0.02), (3001, 0.7, 2, 0.012), (30011, 1.3, 0, 0)]


@pytest.mark.parametrize("divisor,sort", [(1, 1), (1, 0), (2, 1)])
def test_eight_lanes_equal_sixteen(divisor, sort):
    sims = []
    for k, (n, side, blobs, sd) in enumerate(MEMBERS):
        cfg = small_cfg(n=n, side=side, T=2 + k, seed=k + 1)
        if blobs:
            cfg["init"] = dict(kind="blobs", count=blobs, sd=sd)
        st, phys, _ = state_of(cfg)
        sims.append((phys, st))
    ens = Ensemble(sims)
    ens.setTuning(cell_divisor=divisor, sort_variant=sort)
    ens.simulate(3)
    for s, (ph, st) in enumerate(sims[:-1]):
        plain = make_sim(st, ph)
        plain.setTuning(cell_divisor=divisor, sort_variant=sort)
        plain.simulate(SimulationParams.from_physics(ph), 3)
        assert ens.getParticleData(s).tobytes() == plain.getParticleData().tobytes(), MEMBERS[s]
        assert np.array_equal(ens.getNeighborCounts(s), plain.getNeighborCounts()), MEMBERS[s]
        plain.close()
    ens.close()


# blobs whose owners have from none to several hundred partners: the LDS list (24 or 48), the
# wave's list of 192 and its cuts
@pytest.mark.parametrize("n,blobs,sd,far", [(3000, 60, 0.004, 0), (4000, 3, 0.004, 0),
                                            (30000, 40, 0.004, 0), (3000, 12, 0.004, 1)])
@pytest.mark.parametrize("maxc", [1, 16, 32])
def test_wave_edge_selection(orc, n, blobs, sd, far, maxc):
    """`far`: an edge distance beyond one cell, so every graph is the standalone pass's."""
    cfg = small_cfg(n=n, side=1.0, T=2, seed=n + blobs, radius=0.02 if far else 0.05)
    cfg["init"] = dict(kind="blobs", count=blobs, sd=sd)
    st, phys, params = state_of(cfg)
    dist = 0.06 if far else 0.012
    sim = make_sim(st, phys)
    sim.simulate(params, 0)
    got = sim.getParticleData()
    ref = orc.edges(got["pos"], got["ptype"], dist, maxc, mode=1)
    assert np.array_equal(sim.generateProximityGraph(dist, maxc), ref) and len(ref) > 0
    if not far:
        for sort in (0, 1):
            a, b = make_sim(st, phys), make_sim(st, phys)
            for h in (a, b):
                h.setTuning(sort_variant=sort)
            check_step_edges(orc, a, b, params, (dist, maxc), mode=1)
