"""The edges of the step's spread counters, queue segments and grid build:
crowds at the sizes where the 3D-LP queue's segments grow, and grids whose
block totals a scatter block scans one per thread, eight per thread or finds
scanned, give the same states, neighbours and statistics, bit for bit, as the
row step or a coarse grid; agents whose half-planes the branch-free form does
not cover (no radius, T off the powers of two) match the oracle; and host
batches around the staging's pieces give the network's rows.  A step with more
events than the host block holds delivers them all."""
import numpy as np
import pytest

from ecmgenerator_amd.learned import ProposalNet
from ecmgenerator_amd.simulator import Agents, Params, Simulator
from helpers import compare_step, oracle_state, small_scene
from test_gpu_row_step import same

pytestmark = pytest.mark.gpu


def jam(n, seed):
    """A crowd that walks to one point at some 4 agents a square metre."""
    rng = np.random.default_rng(seed)
    half = float(np.sqrt(n / 4.0) / 2.0)
    start = rng.uniform(-half, half, (n, 2)).astype(np.float32)
    goal = np.full((n, 2), half + 25.0, np.float32)
    path = np.stack([start, goal], 1).reshape(-1, 2)
    agents = Agents(start, rng.uniform(0.2, 0.3, n).astype(np.float32), rng.uniform(1.0, 1.6, n).astype(np.float32),
                    np.arange(n, dtype=np.int32) * 2, np.full(n, 2, np.int32), path)
    _, _, obs, _, _ = small_scene(seed, half=half + 5.0, n_rects=4, n_agents=1, side=(1, 3))
    return (-half - 30.0, -half - 30.0, half + 30.0, half + 30.0), obs, agents


def square(box):
    from ecmgenerator_amd import scenarios as S
    return S.empty_square_ecm(*box)


@pytest.mark.parametrize("shape", [(64, 2), (256, 1)])
@pytest.mark.parametrize("n", [63, 64, 65, 4096, 4097, 8193])
def test_queue_segments(n, shape):
    box, obs, agents = jam(n, n)

    def make():
        sim = Simulator(square(box), obs, box, Params(max_agents=n, keep_orca_velocity=True))
        sim.SpawnAgents(agents, validate=False)
        return sim
    row, lane = make(), make()
    lane.set_tuning(knn_block=shape[0], orca_obst_slots=shape[1])
    for _ in range(4):
        row.Update()
        lane.Update()
        same(row, lane)
    assert n < 100 or row.stats()["lp3d"] > n // 10
    row.close()
    lane.close()


# cells of 0.5 m: totals of 64, 256, 1024 and, over three environments, 3072 scan blocks
@pytest.mark.parametrize("shape", [256, 64])
@pytest.mark.parametrize("half,envs", [(120.0, 1), (250.0, 1), (500.0, 1), (500.0, 3)])
def test_fine_grid_equals_coarse(half, envs, shape):
    scenes = [small_scene(7 + e, half=half, n_rects=6, n_agents=400, side=(1, 8)) for e in range(envs)]

    def make(cell):
        box, _, obs, ecm, agents = scenes[0]
        sim = Simulator(ecm, obs, box, Params(max_agents=400 * envs, keep_orca_velocity=True, grid_cell=cell))
        sim.SpawnAgents(agents)
        for box, _, obs, ecm, agents in scenes[1:]:
            sim.SpawnAgents(agents, env=sim.AddEnvironment(ecm, obs, box))
        sim.set_tuning(knn_block=shape)
        return sim
    fine, coarse = make(0.5), make(20.0)
    for _ in range(4):
        fine.Update()
        coarse.Update()
        same(fine, coarse)
    fine.close()
    coarse.close()


@pytest.mark.parametrize("horizon", [2.0, 1.5])
@pytest.mark.parametrize("k,shape", [(5, (64, 2)), (10, (64, 2)), (10, (256, 1)), (16, (256, 2))])
def test_uncovered_half_planes(k, shape, horizon):
    from oracle import oracle_py as O
    box, _, obs, ecm, agents = small_scene(50 + k, half=9.0, n_rects=3, n_agents=260, side=(1, 3))
    agents.radius[::3] = 0.0
    p = Params(max_agents=260, k=k, time_horizon=horizon, keep_orca_velocity=True)
    sim = Simulator(ecm, obs, box, p)
    sim.SpawnAgents(agents, validate=False)
    sim.set_tuning(knn_block=shape[0], orca_obst_slots=shape[1])
    for _ in range(4):
        before = oracle_state(sim)
        ora = O.step(p, before, obs, ecm)
        sim.Update()
        assert not {a: b for a, b in compare_step(sim, before, ora).items() if b}
    sim.close()


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 32768, 32769, 66000])
def test_staged_batches(n):
    net = ProposalNet.load()
    rng = np.random.default_rng(n)
    x = rng.normal(0.0, 1.0, (n, 64)).astype(np.float32)
    x[:, 61:] = 0.0
    y = net.forward(x)
    for a in (0, max(0, n // 2 - 100), max(0, n - 300)):
        assert np.array_equal(y[a:a + 300], net.forward(np.ascontiguousarray(x[a:a + 300])))


@pytest.mark.parametrize("shape", [256, 64])
def test_more_events_than_the_host_block_holds(shape):
    """1,500 agents at their goals beside 500 that walk: the events past the
    host block's 1,024 are copied from the device's list."""
    rng = np.random.default_rng(9)
    n, gone = 2000, 1500
    start = rng.uniform(-60.0, 60.0, (n, 2)).astype(np.float32)
    off = np.where(np.arange(n)[:, None] < gone, 0.5, 40.0).astype(np.float32)
    path = np.stack([start, start + off], 1).reshape(-1, 2).astype(np.float32)
    agents = Agents(start, np.full(n, 0.2, np.float32), np.full(n, 1.3, np.float32),
                    np.arange(n, dtype=np.int32) * 2, np.full(n, 2, np.int32), path)
    box = (-120.0, -120.0, 120.0, 120.0)
    _, _, obs, _, _ = small_scene(3, half=100.0, n_rects=1, n_agents=1, side=(1, 2))
    sim = Simulator(square(box), obs, box, Params(max_agents=n))
    ids = sim.SpawnAgents(agents, validate=False)
    sim.set_tuning(knn_block=shape)
    sim.Update(steps=3)
    active = sim.state()["active"].astype(bool)
    assert not active[ids[:gone]].any() and active[ids[gone:]].all()
    again = sim.SpawnAgents(Agents(start[:gone], agents.radius[:gone], agents.pref_speed[:gone], agents.path_off[:gone],
                                   agents.path_cnt[:gone], path), validate=False)
    assert np.array_equal(np.sort(again), np.sort(ids[:gone]))
    sim.close()
