"""The plain step with 16 lanes per agent (small crowds in the default launch
shape) against the one-agent-per-lane passes (the launch shape with 64-thread
workgroups): every component, the neighbour lists and the statistics must be
equal bit for bit, step after step.  The scenes reach the edges of the row
form: 1 to 16 neighbours, crowds that do not fill a wavefront or fill it by
one, fewer agents than neighbours, agents on one lattice (equal distances,
more candidates than the buffer holds), obstacle lists past 16 and 64 edges,
agents outside the grid box, and several environments."""
import numpy as np
import pytest

from ecmgenerator_amd import scenarios as S
from ecmgenerator_amd.simulator import Agents, Params, Simulator
from helpers import small_scene

pytestmark = pytest.mark.gpu

KEYS = ("position", "velocity", "attraction", "pref_velocity", "active", "orca_velocity")


def same(a, b):
    sa, sb = a.state(), b.state()
    for key in KEYS:
        assert np.array_equal(sa[key], sb[key], equal_nan=True), key
    na, ca = a.neighbors()
    nb, cb = b.neighbors()
    assert np.array_equal(ca, cb) and np.array_equal(na, nb)
    assert np.array_equal(a.replans(), b.replans())
    assert a.stats() == b.stats()


def run_both(make, steps, between=None):
    row, lane = make(), make()
    lane.set_tuning(knn_block=64)
    for it in range(steps):
        if between is not None:
            for sim in (row, lane):
                between(it, sim)
        row.Update()
        lane.Update()
        same(row, lane)
    st = row.stats()
    row.close()
    lane.close()
    return st


@pytest.mark.parametrize("k", [1, 2, 5, 9, 10, 15, 16])
@pytest.mark.parametrize("n", [1, 4, 17, 260])
def test_row_step_equals_lane_step(k, n):
    box, rects, obs, ecm, agents = small_scene(100 * k + n, half=14.0, n_rects=5, n_agents=n, side=(1, 4))

    def make():
        sim = Simulator(ecm, obs, box, Params(max_agents=n + 3, k=k, keep_orca_velocity=True))
        sim.SpawnAgents(agents)
        return sim

    def push(it, sim):
        if it == 3:                              # a state from elsewhere: loose seeds, agents outside the box
            rng = np.random.default_rng(k)
            sim.write("position", rng.uniform(-16.0, 16.0, (n + 3, 2)).astype(np.float32))
    st = run_both(make, 8, push)
    if n == 260:
        assert st["lp3d"] > 0


def test_row_step_lattice_and_long_obstacle_lists():
    box = (-30.0, -30.0, 30.0, 30.0)
    rng = np.random.default_rng(3)
    side = 24
    gx, gy = np.meshgrid(np.arange(side) * 0.5 - 6.0, np.arange(side) * 0.5 - 6.0)
    start = np.stack([gx.ravel(), gy.ravel()], 1).astype(np.float32)
    n = start.shape[0]
    goal = rng.uniform(-25.0, 25.0, (n, 2)).astype(np.float32)
    path = np.stack([start, goal], 1).reshape(-1, 2)
    agents = Agents(start, np.full(n, 0.25, np.float32), np.full(n, 1.3, np.float32),
                    np.arange(n, dtype=np.int32) * 2, np.full(n, 2, np.int32), path)
    for gap, count in ((1.4, 5), (0.9, 9)):       # pillars around the crowd: short and long bucket lists
        c = (np.arange(count) - count // 2) * gap
        rings = [S.rect_ring(x + 8.0, y, 0.2, 0.2) for x in c for y in c]
        xy = np.concatenate(rings).astype(np.float32)
        obs = type(S.rects_to_obstacles([]))(xy, np.arange(len(rings) + 1, dtype=np.int32) * 4)

        def make():
            p = Params(max_agents=n, keep_orca_velocity=True, grid_cell=6.0)
            sim = Simulator(S.empty_square_ecm(*box), obs, box, p)
            sim.SpawnAgents(agents, validate=False)
            return sim
        st = run_both(make, 5)
        assert st["obst_overflow"] > 0 and st["lp3d_big"] > 0


def test_row_step_environments():
    scenes = [small_scene(s, half=10.0 + 4 * s, n_rects=3, n_agents=40 * s + 1, side=(1, 4)) for s in (1, 2, 3)]
    total = sum(sc[4].n for sc in scenes)

    def make():
        box, _, obs, ecm, agents = scenes[0]
        sim = Simulator(ecm, obs, box, Params(max_agents=total, keep_orca_velocity=True))
        sim.SpawnAgents(agents)
        for box, _, obs, ecm, agents in scenes[1:]:
            sim.SpawnAgents(agents, env=sim.AddEnvironment(ecm, obs, box))
        sim.set_graph(True)
        return sim
    run_both(make, 10)
