"""GPU: the graph built inside a step, at the sizes where the force pass's edge lists change
(64 slots of either index per owner, 20 to 64 of them above the owner's index by lanes per
particle, the wave beyond), for the default tuning, both list variants and small grids,
against the oracle's graph of the same state, bit for bit."""

import numpy as np
import pytest

from cellflow_amd import ParticleSimulation, SimulationParams, particles_from_state

pytestmark = pytest.mark.gpu

TUNINGS = [(0, 16, 1), (3, 4, 0), (3, 32, 1), (4, 8, 1), (4, 16, 0)]


@pytest.mark.parametrize("k", [2, 21, 22, 41, 42, 64, 65, 66, 131])
@pytest.mark.parametrize("side", [0.9, 0.1])  # 0.1: two cells per axis, per-pair images
def test_step_edge_lists(orc, k, side):
    """k particles of one type in each of a few clumps of radius 0.004, at rest and without
    forces, so the state of the second step is the one loaded."""
    rng = np.random.default_rng(k)
    at = np.array([[0.05, 0.05, 0.05], [0.25, 0.3, 0.35], [0.6, 0.1, 0.8]])[: 3 if side > 0.5 else 1]
    d = rng.uniform(-0.0023, 0.0023, (len(at), k, 3))
    pos = np.concatenate([(at[:, None] + d).reshape(-1, 3), rng.random((200, 3)) * side])
    ty = np.concatenate([np.zeros(len(at) * k, np.uint32), rng.integers(0, 2, 200)]).astype(np.uint32)
    order = rng.permutation(len(pos))
    pos, ty = pos[order].astype(np.float32), ty[order]
    for variant, lanes, sort in TUNINGS:
        sim = ParticleSimulation(len(pos), 2)
        sim.setForceTable(np.zeros((2, 2), np.float32))
        sim.setRadioByType(np.zeros(2, np.float32))
        sim.setTuning(force_variant=variant, lanes_per_particle=lanes, sort_variant=sort)
        sim.setParticles(particles_from_state(pos, np.zeros_like(pos), ty))
        params = SimulationParams(radius=0.04, ratioWithLFO=0.0, numParticleTypes=2, repulsion=0.0,
                                  attraction=0.0, canvasWidth=side, canvasHeight=side,
                                  canvasDepth=side)
        for maxc in (3, 16, 32):
            sim.simulate(params, 2, edges=(0.012, maxc))
            got = sim.getParticleData()
            ref = orc.edges(got["pos"], got["ptype"], 0.012, maxc, mode=1)
            assert len(ref) > 0
            assert np.array_equal(sim.getStepEdges(), ref), (variant, lanes, maxc)
            assert np.array_equal(sim.getEdges(), ref), (variant, lanes, maxc)
        sim.close()
