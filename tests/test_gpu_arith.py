"""The device code's own arithmetic against the plain operations it stands for,
bit for bit (tests/cpp/arith_check.hip, built with the library): roots and
reciprocals for every mantissa at every exponent they are used at, quotients
over random and extreme pairs, the arc tangent for every float in [0, 1], and
the branch-free half-plane against the branching one over common operands and
at each guard that sends an operand to the latter."""
import ctypes as C
import os

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

LIB = os.path.join(ROOT, "tests", "cpp", "_build", "libarith_check.so")


@pytest.fixture(scope="module")
def lib(native_gpu):
    return C.CDLL(LIB)


def counts(fn, *args):
    out = (C.c_ulonglong * 2)()
    assert fn(*args, out) == 0
    return out[0], out[1]


@pytest.mark.parametrize("what,lo,hi", [("root", -96, 96), ("reciprocal", -60, 60), ("reciprocal of a root", -60, 60)])
def test_every_mantissa(lib, what, lo, hi):
    bad, n = counts(lib.check_unary, ["root", "reciprocal", "reciprocal of a root"].index(what), lo, hi)
    assert bad == 0 and n > 0.99 * (hi - lo) * 2 ** 23


def test_atan_unit(lib):
    assert counts(lib.check_atan) == (0, 0x3f800001)


@pytest.mark.parametrize("seed", [1, 2])
def test_quotients(lib, seed):
    bad, n = counts(lib.check_quot, C.c_uint32(seed), 256)
    assert bad == 0 and n > 2 ** 27


def pairs(kind, T, dt, n=100_000, seed=0):
    """[n, 10]: position, velocity, radius of an agent and of the other."""
    rng = np.random.default_rng(seed)
    f = np.float32
    p = rng.uniform(-100.0, 100.0, (n, 2))
    rel = rng.uniform(-5.0, 5.0, (n, 2))
    v, qv = rng.normal(0.0, 1.0, (2, n, 2))
    r, qr = rng.uniform(0.15, 0.35, (2, n))

    def power(lo, hi, shape):
        return np.exp2(rng.integers(lo, hi + 1, shape)) * rng.choice([1.0, 1.0 + 2.0 ** -23, 2.0 - 2.0 ** -23], shape)
    sign = rng.choice([-1.0, 1.0], (n, 2))
    if kind == "close":                              # half of them colliding
        rel *= 0.1
    elif kind == "scales":
        p[:] = 0.0
        rel = sign * power(-34, 34, (n, 1)) * rng.uniform(0.1, 1.0, (n, 2))
        r = power(-64, 34, n)
        v = v * power(-34, 34, (n, 1))
    elif kind == "tiny components":
        p[:] = 0.0
        rel[:, 0] = np.where(rng.random(n) < 0.2, 0.0, sign[:, 0] * power(-90, -70, n))
        v[:, 1] = qv[:, 1]
    elif kind == "lengths of ones":
        p[:] = 0.0
        rel = np.stack([(2.0 - 2.0 ** -23) * np.exp2(rng.integers(-32, 32, n)), np.zeros(n)], 1)
        rel = np.where(rng.random((n, 1)) < 0.5, rel, rel[:, ::-1]) * sign
    elif kind == "guards":
        p[:] = 0.0
        rel = np.stack([power(-31, -29, n), np.zeros(n)], 1)
        rel[::2, 0] = power(29, 31, n)[::2]
        r, qr = power(-61, -59, n), np.zeros(n)
        r[::3] = power(59, 61, n)[::3]
    elif kind == "beside the leg":                   # the side of the axis within rounding, or no velocity at all
        k = rng.uniform(-2.0, 2.0, (n, 1))
        v = qv + k * rel
        v[::5] = qv[::5]
        v[1::5] = qv[1::5] + rel[1::5] / T           # on the apex of the cut-off disc
    q = (p.astype(f) + rel.astype(f)).astype(f)
    a = np.concatenate([p, v, r[:, None], q, qr[:, None], qv], 1).astype(f)
    if kind in ("guards", "lengths of ones", "scales", "tiny components"):
        a[:, 5:7] = rel.astype(f)
    if kind == "beside the leg":
        a[:, :2], a[:, 5:7] = 0.0, rel.astype(f)
    if kind == "specials":
        special = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1e-45, -1e-39, 3e38, -3e38, 1e-20, 1e20], f)
        hit = rng.random(a.shape) < 0.15
        a[hit] = rng.choice(special, int(hit.sum()))
        a[::7, 5:7] = a[::7, :2]                     # coincident
    return np.ascontiguousarray(a)


@pytest.mark.parametrize("T,dt", [(2.0, 0.1), (0.5, np.float32(1.0 / 3.0)), (2.0 ** 20, 2.0 ** -20),
                                  (2.0 ** -20, 2.0 ** 20)])
@pytest.mark.parametrize("kind", ["common", "close", "scales", "tiny components", "lengths of ones", "guards",
                                  "beside the leg", "specials"])
def test_half_plane_without_branches(lib, kind, T, dt):
    a = pairs(kind, T, dt)
    n = a.shape[0]
    covered = np.zeros(n, np.uint8)
    f = np.float32
    out = (C.c_ulonglong * 2)()
    rc = lib.check_half_plane(C.c_float(T), C.c_float(float(f(1.0) / f(T))), C.c_float(dt),
                              C.c_float(float(f(1.0) / f(dt))), a.ctypes.data_as(C.c_void_p), n, covered.ctypes.data_as(C.c_void_p), out)
    assert rc == 0
    print(f"{kind} T {T} dt {dt}: {out[1]} of {n} without branches, {out[0]} differ", flush=True)
    assert out[0] == 0 and out[1] == covered.sum()
    if kind in ("common", "close") and T == 2.0:
        assert out[1] > 0.99 * n
    bad = ~np.isfinite(a).all(1)
    assert not (covered.astype(bool) & ~np.isfinite(a[:, [0, 1, 5, 6]]).all(1)).any()
    assert kind != "specials" or (bad.any() and not covered[::7][np.isfinite(a[::7]).all(1)].any())
