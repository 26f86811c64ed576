"""A box of another size is another binning, also when the numbers of cells stay the same:
the state is sorted again before anything walks its cells."""

import dataclasses

import numpy as np
import pytest

from cellflow_amd import grid_dims
from helpers import check_step, make_sim, small_cfg, state_of

pytestmark = pytest.mark.gpu

SIDE, RADIUS = 0.46, 0.05  # 9 cells of 0.0501 a side, with 0.009 to spare


def same(a, b):
    return a.tobytes() == b.tobytes()


def resized(params, f):
    """`params` with each side of the box `f` times as long."""
    return dataclasses.replace(params, canvasWidth=params.canvasWidth * f,
                               canvasHeight=params.canvasHeight * f,
                               canvasDepth=params.canvasDepth * f)


def case(n, factor, divisor):
    st, phys, params = state_of(small_cfg(n=n, side=SIDE, T=3, radius=RADIUS, ratio=0.0))
    big = resized(params, factor)
    # the numbers of cells are the same in both boxes
    assert tuple(grid_dims(params, st["rbt"], n, divisor)) == \
        tuple(grid_dims(big, st["rbt"], n, divisor))
    return st, phys, params, big


@pytest.mark.parametrize("sort_variant", [0, 1])
@pytest.mark.parametrize("variant,lanes", [(0, 16), (0, 8), (4, 8)])
@pytest.mark.parametrize("n,factor,divisor", [(3000, 1.06, 1), (30000, 1.06, 1), (3000, 1.03, 2)])
def test_step_in_a_resized_box(orc, n, factor, divisor, variant, lanes, sort_variant):
    """One step (with its graph) after the box grew: as a fresh simulation at that state, and
    as the oracle."""
    st, phys, params, big = case(n, factor, divisor)
    tuning = dict(cell_divisor=divisor, force_variant=variant, lanes_per_particle=lanes,
                  sort_variant=sort_variant)
    with make_sim(st, phys) as sim:
        sim.setTuning(**tuning)
        sim.simulate(params, 3)
        mid, prev = sim.getParticleData(), sim.getNeighborCounts()
        sim.simulate(big, 1, edges=(0.03, 8))
        got, counts, edges = sim.getParticleData(), sim.getNeighborCounts(), sim.getEdges()
    st2 = dict(st, pos=mid["pos"], vel=mid["vel"], type=mid["ptype"], prev=prev)
    with make_sim(st2, phys) as twin:
        twin.setTuning(**tuning)
        twin.simulate(big, 1, edges=(0.03, 8))
        assert same(twin.getParticleData(), got)
        assert np.array_equal(twin.getNeighborCounts(), counts)
        assert np.array_equal(twin.getEdges(), edges)
    phys2 = dict(phys, canvas=[big.canvasWidth, big.canvasHeight, big.canvasDepth])
    ref = orc.step(mid["pos"], mid["vel"], mid["ptype"], prev, phys2, st["table"], st["rbt"],
                   mode=0)
    assert np.array_equal(counts, ref["count"])
    check_step(got, ref, phys2, mid["vel"])
    assert np.array_equal(edges, orc.edges(got["pos"], got["ptype"], 0.03, 8, mode=0))


@pytest.mark.parametrize("factor", [1.06, 0.96])
def test_overlays_and_histogram_in_a_resized_box(orc, factor):
    """No step in the new box: the graph, the mesh and the histogram of the same state."""
    st, phys, params, _ = case(3000, 1.06, 1)
    first, second = (params, resized(params, 1.06)) if factor > 1 else \
        (resized(params, 1.06), params)
    with make_sim(st, phys) as sim:
        sim.simulate(first, 3)
        mid = sim.getParticleData()
        sim.simulate(second, 0)
        sim.generateProximityGraph(0.04, 8)
        sim.generateTriangleMesh(0.03, 8)
        edges, tris = sim.getEdges(), sim.getTriangles()
        hist = sim.pairHistogram(16, 0.05)
        assert same(sim.getParticleData(), mid)
    st2 = dict(st, pos=mid["pos"], vel=mid["vel"], type=mid["ptype"])
    with make_sim(st2, phys) as twin:
        twin.simulate(second, 0)
        assert same(twin.pairHistogram(16, 0.05), hist)
    assert np.array_equal(edges, orc.edges(mid["pos"], mid["ptype"], 0.04, 8, mode=0))
    assert np.array_equal(tris, orc.triangles(mid["pos"], mid["ptype"], 0.03, 8, mode=0))


def test_graph_replays_survive_a_resized_box():
    """Captured step graphs stay valid: many steps in each box, twice, as fresh simulations."""
    st, phys, params, big = case(3000, 1.06, 1)
    with make_sim(st, phys) as sim:
        for box in (params, big, params, big):
            mid, prev = sim.getParticleData(), sim.getNeighborCounts()
            sim.simulate(box, 70)  # two replays of 32 steps, then single ones
            with make_sim(dict(st, pos=mid["pos"], vel=mid["vel"], type=mid["ptype"],
                               prev=prev), phys) as twin:
                twin.simulate(box, 70)
                assert same(twin.getParticleData(), sim.getParticleData())
