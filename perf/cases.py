"""The work that a program has this framework do, as cases that can be timed.

A crowd case is a rollout: a program puts the crowd into a known state
(ecm_sim_write), advances it by some steps with step graphs on and takes the
positions and velocities back, either once at the end or, as a renderer does,
the positions after every step.  A batch case is the same over several
environments of one handle.  The network cases are the learned proposal's
own calls: its forward pass on device and on host data, its loss and gradient
for one batch, and training on samples that the simulator logged.

A rollout begins from the same state in every pass, so that a crowd that has
been stepped many times is still the crowd of the case.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from ecmgenerator_amd import scene as SC
from ecmgenerator_amd.learned import DEFAULT_WEIGHTS, N_IN, N_IN_PAD, N_OUT, N_SLOTS, ProposalNet
from ecmgenerator_amd.scenarios import agent_draws
from ecmgenerator_amd.simulator import Agents, Params, Simulator

HID = 128
THETA = -2.0                        # the threshold stored with the committed weights
POS_WEIGHT, VEL_WEIGHT = 2.0, 1.0   # ProposalNet.train's defaults
VEL_SCALE = 0.5


def listed():
    return [
        # a room with a few hundred people, drawn every frame: launches and latency
        crowd("room", 30.0, 6, 12, 500, read_every=True),
        # c0 of the benchmark: 200 m, 40 obstacles, 5,000 agents
        crowd("c0", 100.0, 40, 15, 5000),
        # c0 with the reference's literal parameters, drawn every step
        crowd("c0 reference", 100.0, 40, 15, 5000, k=5, reference=True, read_every=True),
        # a town square between the benchmark's sizes; k off the defaults, agents off every power of two
        crowd("town", 350.0, 197, 20, 37411, k=7),
        # c1: 1000 m, 400 obstacles, 100,000 agents
        crowd("c1", 500.0, 400, 25, 100000),
        # c2: a million agents in two opposing flows, jammed in the barrier's gaps
        flows("c2 jam", 950000),
        # the same with the learned proposal in front of the LP
        flows("c2 jam learned", 950000, learned=True),
        # c4 in small: independent environments advanced by one handle
        {"name": "24 environments", "kind": "batch", "envs": 24, "k": 10, "steps": 20, "prerun": 20, "map": 5},
        # the network on device buffers, the largest call it takes
        {"name": "forward on the device", "kind": "forward_device", "n": 32768},
        # the network on host data, as an evaluation script calls it
        {"name": "forward from the host", "kind": "forward", "n": 3001},
        # loss and gradient of the default batch, and training on a logged crowd
        {"name": "loss and gradient", "kind": "grad", "n": 8192},
        {"name": "training", "kind": "train", "agents": 9000, "log_steps": 8, "epochs": 4},
    ]


def crowd(name, half, rects, side, agents, k=10, reference=False, read_every=False, learned=False):
    return {"name": name, "kind": "crowd", "half": half, "rects": rects, "side": side, "agents": agents, "k": k,
            "reference": reference, "read_every": read_every, "learned": learned, "steps": 20, "prerun": 20}


def flows(name, agents, learned=False):
    return {"name": name, "kind": "flows", "agents": agents, "k": 10, "reference": False, "read_every": False,
            "learned": learned, "steps": 20, "prerun": 150}


def draw(rng):
    what = rng.random()
    if what < 0.65:
        agents = int(round(math.exp(rng.uniform(math.log(300), math.log(150000)))))
        density = math.exp(rng.uniform(math.log(0.05), math.log(0.2)))
        half = max(20.0, float(round(math.sqrt(agents / density) / 2)))
        rects = int(min(400, 4 * half * half / 250.0) * rng.uniform(0.3, 1.0))
        k = rng.choice([10, 10, 10, 5, 5, 1, 3, 7, 12, 16])
        c = crowd("", half, rects, rng.choice([12, 15, 20, 25]), agents, k=k, reference=rng.random() < 0.2,
                  read_every=rng.random() < 0.3, learned=k == 10 and rng.random() < 0.15)
        c["steps"] = rng.choice([10, 16, 20, 25])
    elif what < 0.72:
        c = flows("", int(rng.uniform(200000, 950000)), learned=rng.random() < 0.25)
        c["prerun"] = int(rng.uniform(20, 150))
    elif what < 0.80:
        c = {"kind": "batch", "envs": rng.randint(2, 24), "k": rng.choice([10, 5]), "steps": 20, "prerun": 20,
             "map": rng.randint(1, 1 << 20)}
    elif what < 0.87:
        c = {"kind": "forward_device", "n": int(round(math.exp(rng.uniform(0.0, math.log(32768)))))}
    elif what < 0.91:
        c = {"kind": "forward", "n": int(round(math.exp(rng.uniform(math.log(30), math.log(60000)))))}
    elif what < 0.96:
        c = {"kind": "grad", "n": int(round(math.exp(rng.uniform(math.log(64), math.log(16384)))))}
    else:
        c = {"kind": "train", "agents": rng.randint(2000, 9000), "log_steps": rng.randint(2, 8),
             "epochs": rng.randint(1, 4)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
def params_of(case, n):
    p = Params.reference(max_agents=n) if case.get("reference") else Params(max_agents=n)
    p.k = case["k"]
    return p


@functools.lru_cache(maxsize=1)
def flow_map():
    """The c2 map with a planned route for each of a million people: what a
    program loads once.  Who walks, how fast and how large is the seed's."""
    sc, agents, _ = SC.generate(2, seed=1)
    return sc, agents


def rollout(sim, case):
    """A spawned simulation some way into its run, the state its rollouts begin from and its host buffers."""
    sim.set_graph(True)
    net = None
    if case.get("learned"):
        net = ProposalNet.load()
        sim.set_learned(net, THETA)
    for _ in range(case["prerun"]):
        sim.Update()
    s = {"case": case, "sim": sim, "net": net}
    for name in ("position", "velocity"):
        s[name] = host_buffer(sim.max_agents)           # where the program reads to
        s[name + "0"] = host_buffer(sim.max_agents)     # the state it sets
        sim.read(name, out=s[name + "0"])
    return s


def host_buffer(n):
    """A page-locked array of n points, as a program that reads back often keeps one."""
    return torch.empty((n, 2), dtype=torch.float32, pin_memory=True).numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "crowd":
        sc, agents, _ = SC.generate_box(case["half"], case["rects"], 2, case["side"], case["agents"], seed=seed + 1)
        sim = Simulator(sc.ecm(), sc.obstacles(), sc.box, params_of(case, agents.n), planner=sc)
        sim.SpawnAgents(agents)
        return rollout(sim, case)
    if kind == "flows":
        sc, pool = flow_map()
        rng = np.random.default_rng(seed)
        who = np.sort(rng.permutation(pool.n)[:case["agents"]])
        radius, speed = agent_draws(rng, who.size)
        agents = Agents(pool.start[who], radius, speed, pool.path_off[who], pool.path_cnt[who], pool.path_xy)
        sim = Simulator(sc.ecm(), sc.obstacles(), sc.box, params_of(case, agents.n), planner=sc)
        sim.SpawnAgents(agents)
        return rollout(sim, case)
    if kind == "batch":
        rng = np.random.default_rng(seed)
        made = []
        for half, rects, n in batch_sizes(case):
            made.append(SC.generate_box(half, rects, 2, 15, n, seed=int(rng.integers(1, 1 << 62)))[:2])
        sc, agents = made[0]
        sim = Simulator(sc.ecm(), sc.obstacles(), sc.box, params_of(case, sum(a.n for _, a in made)), planner=sc)
        sim.SpawnAgents(agents)
        for sc, agents in made[1:]:
            env = sim.AddEnvironment(sc.ecm(), sc.obstacles(), sc.box, planner=sc)
            sim.SpawnAgents(agents, env=env)
        return rollout(sim, case)
    if kind == "forward_device":
        x = torch.from_numpy(samples(seed, case["n"])[0]).cuda()
        y = torch.empty((case["n"], N_OUT), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        return {"case": case, "net": ProposalNet.load(), "x": x, "y": y}
    if kind == "forward":
        return {"case": case, "net": ProposalNet.load(), "x": samples(seed, case["n"])[0]}
    if kind == "grad":
        return {"case": case, "net": ProposalNet.load(), "batch": samples(seed, case["n"])}
    # training: a crowd's samples, taken as one batch, since the order they are logged in is not fixed
    half = math.sqrt(case["agents"] / 0.15) / 2
    sc, agents, _ = SC.generate_box(float(round(half)), 60, 2, 15, case["agents"], seed=seed + 1)
    sim = Simulator(sc.ecm(), sc.obstacles(), sc.box, Params(max_agents=agents.n), planner=sc)
    sim.SpawnAgents(agents)
    net = ProposalNet(seed=seed)
    net.reserve(case["agents"] * case["log_steps"])
    for _ in range(case["log_steps"]):
        sim.log_step(net)
        sim.Update(steps=3)
    sim.close()
    return {"case": case, "net": net, "start": net.get_params(), "n": net.dataset_size()}


def batch_sizes(case):
    """(half side, rectangles, agents) of each environment of a batch case."""
    rng = np.random.default_rng(case["map"])
    out = []
    for _ in range(case["envs"]):
        half = float(np.round(rng.uniform(30.0, 120.0)))
        n = min(int(round(float(np.exp(rng.uniform(np.log(200.0), np.log(5000.0)))))), int(0.2 * 4 * half * half))
        out.append((half, min(int(rng.integers(5, 60)), int(4 * half * half / 250.0)), n))
    return out


def samples(seed, n):
    """Feature rows as a crowd gives them, with label words and LP velocities: neighbours within some 6 m, zeros past
    their count, walls further off, walking speeds."""
    rng = np.random.default_rng(seed)
    x = np.zeros((n, N_IN_PAD), np.float32)
    cnt = np.minimum(rng.integers(3, 14, n), 10)
    near = np.arange(10)[None, :] < cnt[:, None]
    rel = rng.normal(0.0, 0.6, (n, 10, 4)).astype(np.float32)
    x[:, :40] = (rel * near[:, :, None]).reshape(n, 40)
    walls = np.arange(4)[None, :] < rng.integers(0, 5, n)[:, None]
    x[:, 40:56] = (rng.normal(0.0, 1.5, (n, 4, 4)) * walls[:, :, None]).reshape(n, 16)
    x[:, 56:60] = rng.normal(0.0, 0.45, (n, 4))
    x[:, 60] = 4.0 * rng.uniform(0.2, 0.3, n)
    x[:, N_IN:] = 0.0
    np.clip(x, -8.0, 8.0, out=x)
    has = np.concatenate([near, walls], axis=1)
    active = has & (rng.random((n, N_SLOTS)) < 0.15)
    bit = (1 << np.arange(N_SLOTS)).astype(np.uint32)
    label = (active * bit).sum(1).astype(np.uint32) | ((has * bit).sum(1).astype(np.uint32) << 16) | np.uint32(1 << 30)
    v = rng.normal(0.0, 0.9, (n, 2)).astype(np.float32)
    return np.ascontiguousarray(x), label.astype(np.uint32), v


# --------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    net = state.get("net")
    if kind == "forward_device":
        net.forward_device(state["x"].data_ptr(), case["n"], state["y"].data_ptr())
        return state["y"]
    if kind == "forward":
        return net.forward(state["x"])
    if kind == "grad":
        loss, grad = net.loss_grad(*state["batch"], pos_weight=POS_WEIGHT, vel_weight=VEL_WEIGHT)
        return {"loss": loss, "grad": grad}
    if kind == "train":
        net.set_params(state["start"])
        losses = net.train(case["epochs"], batch=state["n"])
        return {"losses": losses, "params": net.get_params()}
    sim = state["sim"]
    sim.write("position", state["position0"])
    sim.write("velocity", state["velocity0"])
    if case.get("read_every"):
        for _ in range(case["steps"]):
            sim.Update()
            sim.GetPositionData(out=state["position"])
    else:
        sim.Update(steps=case["steps"])
        sim.GetPositionData(out=state["position"])
    sim.read("velocity", out=state["velocity"])
    return {"position": state["position"], "velocity": state["velocity"]}


# -------------------------------------------------------------------- work
#: of one sample: 2 x (64 x 128 + 2 x 128 x 128 + 128 x 16)
NET_FLOPS = 2.0 * (N_IN_PAD * HID + 2 * HID * HID + HID * N_OUT)
NET_PARAMS = N_IN_PAD * HID + 2 * HID * HID + HID * N_OUT + 3 * HID + N_OUT
#: path points of an agent in these maps, on average
PATH_POINTS = 5.0


def work(case):
    kind = case["kind"]
    n = case.get("n", 0)
    if kind in ("forward_device", "forward"):
        return {"bytes": n * (N_IN_PAD + N_OUT) * 4.0 + NET_PARAMS * 2.0, "flops": NET_FLOPS * n}
    if kind == "grad":
        return {"bytes": n * (N_IN_PAD * 4 + 12.0) + NET_PARAMS * 8.0, "flops": 3 * NET_FLOPS * n}
    if kind == "train":
        n = case["agents"] * case["log_steps"]
        return {"bytes": case["epochs"] * (n * (N_IN_PAD * 2 + 12.0) + NET_PARAMS * 16.0),
                "flops": 3 * NET_FLOPS * n * case["epochs"]}
    agents = sum(b[2] for b in batch_sizes(case)) if kind == "batch" else case["agents"]
    # a step reads each agent's state and path and writes its new state; the arithmetic: a half-plane for each of k
    # neighbours and one pass of the LP over them
    steps = agents * case["steps"]
    flops = steps * (case["k"] * 120.0 + case["k"] * case["k"] * 10.0)
    if case.get("learned"):
        flops += steps * NET_FLOPS
    return {"bytes": steps * (58.0 + 8.0 * PATH_POINTS) + agents * 32.0, "flops": flops}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """The network's outputs in 64 bits.  A rollout has no such value: its result is the binary32 one (each neighbour
    and each LP constraint is taken or left by a comparison of binary32 numbers, and a crowd in 64 bits parts from it
    within a few steps); neither has training, whose samples the simulator makes."""
    kind = case["kind"]
    if kind not in ("forward_device", "forward", "grad"):
        return None
    x, label, v = samples(seed, case["n"])
    with np.load(DEFAULT_WEIGHTS, allow_pickle=False) as z:
        p = torch.from_numpy(z["params"].astype(np.float64))
    p.requires_grad_(kind == "grad")
    h, at = torch.from_numpy(x.astype(np.float64)), 0
    for rows, cols in ((HID, N_IN_PAD), (HID, HID), (HID, HID), (N_OUT, HID)):
        w, b = p[at:at + rows * cols].reshape(rows, cols), p[at + rows * cols:at + rows * cols + rows]
        at += rows * cols + rows
        h = h @ w.T + b
        if rows == HID:
            h = torch.nn.functional.silu(h)
    if kind != "grad":
        return h.detach()
    bits = torch.arange(N_SLOTS)
    word = torch.from_numpy(label.astype(np.int64))[:, None]
    t, valid = ((word >> bits) & 1).double(), ((word >> (bits + 16)) & 1).double()
    lg, ev = h[:, :N_SLOTS], h[:, N_SLOTS:] - torch.from_numpy(v.astype(np.float64)) * VEL_SCALE
    softplus = torch.nn.functional.softplus
    bce = t * POS_WEIGHT * softplus(-lg) + (1.0 - t) * softplus(lg)
    loss = ((valid * bce).sum() + 0.5 * VEL_WEIGHT * (ev * ev).sum()) / case["n"]
    loss.backward()
    return {"loss": float(loss.detach()), "grad": p.grad}
