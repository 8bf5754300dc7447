"""How a step is put on the stream: with graphs on, a step that finds the
stream idle replays its graph (the autotuner's samples among them, and a step
behind one whose events overflowed the host block), and a crowd whose count
moves around a multiple of 4,096 does not capture its graphs anew.  The
autotuner finds the form with 16 lanes per agent from any launch shape, and a
crowd that crosses the form's limits, or whose map has long obstacle lists,
gives the same steps as one that never takes it."""
import numpy as np
import pytest

from ecmgenerator_amd import scenarios as S
from ecmgenerator_amd.simulator import Agents, Obstacles, Params, Simulator
from helpers import small_scene
from test_gpu_row_step import same

pytestmark = pytest.mark.gpu


def walkers(n, seed, half=60.0, far=1000.0, extra=0, k=10, keep=False):
    """n agents on their way to goals far outside: none arrives."""
    rng = np.random.default_rng(seed)
    start = rng.uniform(-half, half, (n, 2)).astype(np.float32)
    path = np.stack([start, start * 0 + np.float32(far)], 1).reshape(-1, 2).astype(np.float32)
    agents = Agents(start, rng.uniform(0.2, 0.3, n).astype(np.float32), rng.uniform(1.0, 1.6, n).astype(np.float32),
                    np.arange(n, dtype=np.int32) * 2, np.full(n, 2, np.int32), path)
    box, _, obs, ecm, _ = small_scene(seed, half=half + 40.0, n_rects=3, n_agents=1, side=(1, 3))
    sim = Simulator(ecm, obs, box, Params(max_agents=n + extra, k=k, keep_orca_velocity=keep))
    sim.SpawnAgents(agents, validate=False)
    return sim, agents


def test_autotune_times_graph_replays():
    sim, _ = walkers(1500, 3)
    sim.set_graph(True)
    sim.Update()
    steps, replays = sim.stats()["steps"], sim.graph_counts()[0]
    sim.autotune(2)
    assert sim.graph_counts()[0] - replays == sim.stats()["steps"] - steps > 20
    sim.close()


def test_step_behind_an_event_overflow_replays():
    """2,000 agents outside every cell ask for a path each step: the step waits for the device's list."""
    sim, agents = walkers(2000, 4, half=20.0)
    sim.set_graph(True)
    sim.write("position", np.full((2000, 2), 500.0, np.float32) + agents.start)
    sim.Update(steps=4)
    assert sim.replans().size == 2000
    assert sim.graph_counts()[0] == 4
    sim.close()


def test_moving_count_keeps_the_graphs():
    sim, agents = walkers(4100, 5, extra=8)
    sim.set_graph(True)
    ids = list(np.flatnonzero(sim.GetActiveFlags()))
    one = Agents(agents.start[:1], agents.radius[:1], agents.pref_speed[:1], agents.path_off[:1], agents.path_cnt[:1],
                 agents.path_xy[:2])
    captures = 0
    for it in range(12):                         # 4,100, then 4,090 and back, two steps each
        if it % 4 == 2:
            for i in ids[-10:]:
                sim.DestroyAgent(int(i))
            ids = ids[:-10]
        elif it % 4 == 0 and it:
            ids += [int(sim.SpawnAgents(one, validate=False)[0]) for _ in range(10)]
        sim.Update()
        sim.GetPositionData()
        if it == 4:                              # both parities, entered from the slots and from the last step
            captures = sim.graph_counts()[1]
    assert sim.GetNumAgents() == 4090
    assert sim.graph_counts() == (12, captures)
    sim.close()


@pytest.mark.parametrize("shape", [(64, 1), (16, 4), (128, 2), (256, 2)])
def test_autotune_finds_the_row_step(shape):
    """500 agents, three times as fast with 16 lanes each."""
    sim, _ = walkers(500, 6)
    sim.set_graph(True)
    sim.set_tuning(knn_block=shape[0], orca_obst_slots=shape[1])
    sim.Update()
    t = sim.autotune(3)
    assert (t["knn_block"], t["orca_obst_slots"]) == (256, 2)
    sim.close()


@pytest.mark.parametrize("limit,k", [(112000, 5), (16000, 10)])
def test_crossing_a_limit(limit, k):
    """The step's limit at k 5 and the attraction pass's: past it, an eighth below it and past it again, with graphs."""
    n, back = limit - 10, limit - limit // 8 - 10
    sims = []
    for shape in (256, 64):
        sim, agents = walkers(n, 8, half=float(np.sqrt(n / 0.3) / 2), extra=limit // 8 + 100, k=k, keep=True)
        sim.set_tuning(knn_block=shape)
        sim.set_graph(True)
        sims.append(sim)

    def part(m):
        return Agents(agents.start[:m] + np.float32(0.4), agents.radius[:m], agents.pref_speed[:m], agents.path_off[:m],
                      agents.path_cnt[:m], agents.path_xy)
    for act in ("", "", "over", "", "below", "", "over", ""):
        for sim in sims:
            have = sim.GetNumAgents()
            if act == "over":
                sim.SpawnAgents(part(limit + 20 - have), validate=False)
            elif act == "below":
                for i in np.flatnonzero(sim.GetActiveFlags())[:have - back]:
                    sim.DestroyAgent(int(i))
            sim.Update()
        assert sims[0].GetNumAgents() in (n, limit + 20, back)
        same(*sims)
    for sim in sims:
        sim.close()


def test_timing_names_the_form():
    sim, _ = walkers(300, 9)
    sim.set_timing(True)
    for shape, row in (((256, 2), True), ((64, 2), False), ((256, 1), False), ((256, 2), True)):
        sim.set_tuning(knn_block=shape[0], orca_obst_slots=shape[1])
        sim.Update()
        t = sim.last_timing()
        assert sim.last_step_row() == row and len(t) == 6
        assert t[1] >= t[5] > 0.0
    sim.close()


def test_long_obstacle_lists_in_a_large_crowd():
    """30,000 agents and a spot of pillars with several hundred edges within range of one point: every wavefront of
    the row step holds room for the longest list."""
    n, half = 30000, 200.0
    rng = np.random.default_rng(10)
    start = rng.uniform(-half, half, (n, 2)).astype(np.float32)
    start[:3000] = rng.uniform(-8.0, 8.0, (3000, 2))
    goal = rng.uniform(-half, half, (n, 2)).astype(np.float32)
    agents = Agents(start, rng.uniform(0.15, 0.25, n).astype(np.float32), rng.uniform(1.0, 1.6, n).astype(np.float32),
                    np.arange(n, dtype=np.int32) * 2, np.full(n, 2, np.int32), np.stack([start, goal], 1).reshape(-1, 2))
    c = (np.arange(9) - 4) * 1.0
    rings = [S.rect_ring(x, y, 0.2, 0.2) for x in c for y in c]
    obs = Obstacles(np.concatenate(rings).astype(np.float32), np.arange(len(rings) + 1, dtype=np.int32) * 4)
    box = (-half - 5.0, -half - 5.0, half + 5.0, half + 5.0)
    sims = []
    for shape in (256, 64):
        sim = Simulator(S.empty_square_ecm(*box), obs, box, Params(max_agents=n, keep_orca_velocity=True))
        sim.SpawnAgents(agents, validate=False)
        sim.set_tuning(knn_block=shape)
        sims.append(sim)
    for _ in range(4):
        for sim in sims:
            sim.Update()
        same(*sims)
    assert sims[0].stats()["lp3d_big"] > 100
    for sim in sims:
        sim.close()
