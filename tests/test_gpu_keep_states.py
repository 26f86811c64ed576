"""GPU: the gradient with every state kept (short rollouts) against the one that recomputes
its segments from checkpoints (when keeping all would take over 16 times the buffers the
caller's interval takes): every output bit for bit, with force-kernel lists and with the walk's."""

import numpy as np
import pytest

from helpers import make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant,lanes", [(0, 16), (0, 8), (3, 8)])
def test_kept_states_equal_recomputed_ones(variant, lanes):
    st, phys, params = state_of(small_cfg(n=1999, side=0.5, T=3, delta_t=0.001))
    target = np.linspace(0.0, 8.0, 16)
    steps = 403
    got = []
    # 403 steps: intervals 9 and 12 recompute (403 states are over 16 times theirs), 403 and
    # 100 keep every state
    for every in (403, 100, 12, 9):
        sim = make_sim(st, phys)
        sim.setTuning(force_variant=variant, lanes_per_particle=lanes)
        loss, hist, table, ratio = sim.rolloutGrad(params, steps, every, 16, 0.1, target)
        end = sim.getParticleData()
        got.append((loss, hist.tobytes(), table.tobytes(), ratio, end["pos"].tobytes(),
                    end["vel"].tobytes(), sim.getNeighborCounts().tobytes()))
        # the same call again from the same state, on the buffers of the first
        sim.setParticles(make_sim(st, phys).getParticleData())
        again = sim.rolloutGrad(params, steps, every, 16, 0.1, target)
        assert again[0] == loss and again[2].tobytes() == table.tobytes()
        sim.close()
    assert np.isfinite(got[0][0]) and np.abs(np.frombuffer(got[0][2])).max() > 0
    assert all(g == got[0] for g in got[1:])
