"""GPU: tiles of the step's tile sort that several blocks share (more than 1,024 members),
against the counting sort, which knows no tiles: states, counts, order and graphs bit for bit."""

import numpy as np
import pytest

from helpers import make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu

# corner box (as parts of the side) that holds everything: one cell, one row, one plane's
# rows, a block of cells; sizes around a tile's capacity and a part, and past one round of
# the helper blocks' first parts
BOXES = {"cell": (0.02, 0.02, 0.02), "row": (0.9, 0.02, 0.02), "plane": (0.9, 0.9, 0.02),
         "block": (0.25, 0.25, 0.25)}


SIZES = [1023, 1025, 1537, 5000]


@pytest.mark.parametrize("box,n", [(b, n) for b in sorted(BOXES) for n in SIZES] +
                         [(b, 24001) for b in ("block", "plane", "row")])
def test_shared_tiles_equal_the_counting_sort(box, n):
    st, phys, params = state_of(small_cfg(n=n, side=1.0, T=3, seed=n))
    rng = np.random.default_rng(n)
    st["pos"] = (rng.random((n, 3)) * np.array(BOXES[box])).astype(np.float32)
    st["vel"] = (0.5 * rng.standard_normal((n, 3))).astype(np.float32)
    out = []
    for sort in (0, 1):
        sim = make_sim(st, phys)
        sim.setTuning(sort_variant=sort)
        got = []
        for _ in range(2):  # crowded, then spread by a step or two
            sim.simulate(params, 2, edges=(0.01, 4))
            got += [sim.getParticleData().tobytes(), sim.getNeighborCounts().tobytes(),
                    sim.getEdges().tobytes(), sim.getStepEdges().tobytes(),
                    sim.getSortOrder()[1].tobytes()]
        out.append(got)
        sim.close()
    assert out[0] == out[1]
