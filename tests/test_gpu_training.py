"""The training kernels at the edges of their tiles: loss and gradient against
the oracle for batches that end inside a 32-sample tile, a 64-sample step and
a chunk of the weight gradients; one Adam step of a whole dataset against
numpy; and the weights the Adam step repacks against freshly packed ones.

Tolerance of the gradient: the oracle rounds to BF16 where the kernels do, so
only a value that lands on the other side of a BF16 rounding differs by more
than FP32 rounding.  One of a sample's 128 activations doing so moves a
gradient tensor by 2^-8 / sqrt(128) of its norm, 3.5e-4; three of them in the
same sample stay below 2e-3."""
import ctypes as C

import numpy as np
import pytest

from ecmgenerator_amd.learned import ProposalNet
from ecmgenerator_amd.simulator import Params, Simulator
from helpers import small_scene
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


def batch(n, seed):
    rng = np.random.default_rng(seed)
    x = np.clip(rng.normal(0.0, 0.8, (n, 64)), -8, 8).astype(np.float32)
    x[:, 61:] = 0.0
    valid = rng.integers(0, 1 << 14, n).astype(np.uint32)
    label = (valid & rng.integers(0, 1 << 14, n).astype(np.uint32)) | (valid << np.uint32(16))
    return x, label.astype(np.uint32), rng.normal(0.0, 1.0, (n, 2)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 33, 64, 65, 129, 1000, 8193, 12289])
def test_gradient_at_tile_edges(n):
    net = ProposalNet(seed=n)
    x, label, v = batch(n, n)
    loss, grad = net.loss_grad(x, label, v, pos_weight=2.0, vel_weight=0.7)
    again = net.loss_grad(x, label, v, pos_weight=2.0, vel_weight=0.7)
    lo, go = M.loss_grad(net.get_params(), x, label, v, pos_weight=2.0, vel_weight=0.7)
    assert loss == again[0] and np.array_equal(grad, again[1])
    assert abs(loss - lo) <= 1e-4 * abs(lo)
    got, want = M.unflatten(grad), M.unflatten(go)
    for name in want:
        err = np.linalg.norm(got[name] - want[name]) / max(np.linalg.norm(want[name]), 1e-12)
        assert err < 2e-3, (name, err)
    net.close()


def test_adam_step_and_repacked_weights():
    box, _, obs, ecm, agents = small_scene(5, n_agents=300)
    sim = Simulator(ecm, obs, box, Params(max_agents=agents.n))
    sim.SpawnAgents(agents)
    net = ProposalNet(seed=3)
    net.reserve(4000)
    for _ in range(6):
        sim.log_step(net)
    sim.close()
    n = net.dataset_size()
    p0 = net.get_params()
    x, label, v = net.read(0, n)
    loss, g = net.loss_grad(x, label, v)
    losses = net.train(1, batch=n, lr=1e-3)
    assert abs(losses[0] - loss) <= 1e-5 * abs(loss)
    p1 = net.get_params()
    big = np.abs(g) > 1e-4 * np.abs(g).max()
    step = 1e-3 * g / (np.abs(g) + 1e-8)          # the first step's moments are g and g^2
    assert np.abs((p0 - p1) - step)[big].max() < 1e-3 * 1e-3 + 2.0 ** -24
    assert np.array_equal(p0[g == 0.0], p1[g == 0.0])
    net.train(2, batch=max(64, n // 3), seed=1)
    fresh = ProposalNet(params=net.get_params())
    a, b = net.loss_grad(x, label, v), fresh.loss_grad(x, label, v)
    assert a[0] == b[0] and np.array_equal(a[1], b[1])
    assert np.array_equal(net.forward(x), fresh.forward(x))
    net.close()
    fresh.close()


def test_forward_from_unaligned_rows():
    """Device rows that start on a 16-byte boundary, and 4 and 8 bytes past one."""
    hip = C.CDLL("libamdhip64.so")
    net = ProposalNet.load()
    dx, dy = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(dx), C.c_size_t(200 * 256 + 16)) == 0
    assert hip.hipMalloc(C.byref(dy), C.c_size_t(200 * 64)) == 0
    try:
        for n in (1, 33, 200):
            x = batch(n, n)[0]
            want = net.forward(x)
            for off in (0, 4, 8):
                at = C.c_void_p(dx.value + off)
                assert hip.hipMemcpy(at, x.ctypes.data_as(C.c_void_p), C.c_size_t(x.nbytes), 1) == 0
                net.forward_device(at.value, n, dy.value)
                y = np.empty((n, 16), np.float32)
                assert hip.hipMemcpy(y.ctypes.data_as(C.c_void_p), dy, C.c_size_t(y.nbytes), 2) == 0
                assert np.array_equal(y, want), (n, off)
    finally:
        hip.hipFree(dx)
        hip.hipFree(dy)
        net.close()
