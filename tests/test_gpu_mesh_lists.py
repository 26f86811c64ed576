"""The triangle mesh's owner lists at the sizes where their handling changes, against the
oracle (bit for bit: index work): clumps of one type with k members, so an owner's LDS list
is just full, just over (the whole wave selects), or many times over; the 64-triangle cap; a
wave's 64 owners with and without triangles; and reaches of one cell and of several."""

import numpy as np
import pytest

from cellflow_amd import ParticleSimulation, SimulationParams, particles_from_state

pytestmark = pytest.mark.gpu


def mesh_sim(k, side, seed):
    """Clumps of k particles of one type and radius 0.004, 0.1 apart, indices shuffled, among
    single particles of the other type."""
    rng = np.random.default_rng([k, seed])
    sites = np.stack(np.meshgrid(*[np.arange(0.05, side, 0.1)] * 3), -1).reshape(-1, 3)
    clumps = sites[: max(1, min(len(sites) // 2, 700 // k))]
    d = rng.uniform(-0.0023, 0.0023, (len(clumps), k, 3))
    pos = np.concatenate([(clumps[:, None] + d).reshape(-1, 3), sites])
    ty = np.concatenate([np.zeros(len(clumps) * k, np.uint32), np.ones(len(sites), np.uint32)])
    order = rng.permutation(len(pos))
    pos, ty = pos[order].astype(np.float32), ty[order]
    sim = ParticleSimulation(len(pos), 2)
    sim.setForceTable(np.zeros((2, 2), np.float32))
    sim.setRadioByType(np.zeros(2, np.float32))
    sim.setParticles(particles_from_state(pos, np.zeros_like(pos), ty))
    sim.simulate(SimulationParams(radius=0.04, ratioWithLFO=0.0, numParticleTypes=2,
                                  canvasWidth=side, canvasHeight=side, canvasDepth=side), 0)
    return sim, pos, ty


@pytest.mark.parametrize("k", [1, 2, 3, 12, 13, 24, 25, 26, 64, 65, 193, 257])
@pytest.mark.parametrize("dist", [0.008, 0.1])
def test_mesh_list_sizes(orc, k, dist):
    sim, pos, ty = mesh_sim(k, 0.5, 7)
    for maxc in (2, 12, 32):
        t = sim.generateTriangleMesh(dist, maxc)
        assert np.array_equal(t, orc.triangles(pos, ty, dist, maxc, mode=1)), maxc
    assert (len(t) > 0) == (k > 2 or dist > 0.05)  # 0.1 joins neighbouring sites
    sim.close()
