"""Edges of the proposal network's calls: output rows that overlap the input
rows on the device, and a handle's first host batch against its later ones."""
import ctypes as C

import numpy as np
import pytest

from ecmgenerator_amd.learned import ProposalNet

pytestmark = pytest.mark.gpu

ROW_IN, ROW_OUT = 256, 64            # bytes of a sample's features and outputs


def rows(seed, n):
    x = np.random.default_rng(seed).normal(0.0, 1.0, (n, 64)).astype(np.float32)
    x[:, 61:] = 0.0
    return x


@pytest.mark.parametrize("n", [1, 33, 5000, 32768])
def test_forward_device_over_its_input(n):
    """y at x's start, one output row before it, one float into it, over its last row and just behind it."""
    hip = C.CDLL("libamdhip64.so")
    net = ProposalNet.load()
    x = rows(n, n)
    want = net.forward(x)
    buf = C.c_void_p()
    assert hip.hipMalloc(C.byref(buf), C.c_size_t(n * (ROW_IN + ROW_OUT) + 2 * ROW_OUT)) == 0
    x_at = buf.value + ROW_OUT
    try:
        for off in (0, -ROW_OUT, 4, n * ROW_IN - ROW_OUT, n * ROW_IN):
            assert hip.hipMemcpy(C.c_void_p(x_at), x.ctypes.data_as(C.c_void_p), C.c_size_t(x.nbytes), 1) == 0
            net.forward_device(x_at, n, x_at + off)
            y = np.empty((n, 16), np.float32)
            assert hip.hipMemcpy(y.ctypes.data_as(C.c_void_p), C.c_void_p(x_at + off), C.c_size_t(y.nbytes), 2) == 0
            assert np.array_equal(y, want), off
    finally:
        hip.hipFree(buf)
        net.close()


@pytest.mark.parametrize("n", [1, 511, 512, 513, 2049])
def test_first_host_call_equals_later_ones(n):
    """A handle's first host call, with few rows through ordinary memory, and the later ones, through page-locked."""
    x = rows(n, n)
    rng = np.random.default_rng(n)
    label = rng.integers(0, 1 << 14, n).astype(np.uint32) | np.uint32(0x3fff << 16)
    v = rng.normal(0.0, 0.9, (n, 2)).astype(np.float32)
    more = rows(n + 1, n + 3000)
    for first in ("forward", "loss_grad"):
        net = ProposalNet.load()
        got = {"forward": [], "loss_grad": []}
        for what in (first, "forward", "loss_grad", "forward", "loss_grad"):
            got[what].append(net.forward(x) if what == "forward" else net.loss_grad(x, label, v))
            if len(got[what]) == 2:
                assert np.array_equal(net.forward(more)[-7:], net.forward(np.ascontiguousarray(more[-7:])))
        assert all(np.array_equal(y, got["forward"][0]) for y in got["forward"])
        assert all(a == got["loss_grad"][0][0] and np.array_equal(g, got["loss_grad"][0][1])
                   for a, g in got["loss_grad"])
        net.close()
