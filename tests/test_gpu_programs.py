"""The interpreter's programs against the same gates in numpy, FP64, at the
sizes where their shape changes: states below, at and above one tile and one
workgroup, whole-state and pass-by-pass launches, 8 and 16 amplitudes per
thread; with the library's tuning and with row-scaled gates.

A gate rounds an amplitude at most 16 times (a 2x2 product and the phases
merged with it) and no gate here has a norm above 1, so none enlarges an error.
The two gates that are not unitary (least singular value 1/2) can halve the
state's norm once each, and with it twice the relative error; a factor 4 is left
for the phases' and rotations' coefficients: 16 eps per gate times 2^4."""
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)
X = np.array([[0, 1], [1, 0]])
Y = np.array([[0, -1j], [1j, 0]])
Z = np.diag([1, -1])
T = np.diag([1, np.exp(0.25j * np.pi)])


def _u3(r):
    t, p, q = r.uniform(0, 2 * np.pi, 3)
    return np.array([[np.cos(t / 2), -np.exp(1j * q) * np.sin(t / 2)],
                     [np.exp(1j * p) * np.sin(t / 2), np.exp(1j * (p + q)) * np.cos(t / 2)]])


def _gates(n, r):
    """Every kind of gate on free, controlled and anti-controlled targets."""
    out = []
    for b in range(n):
        out.append((b, 0, 0, (H, X, Y, _u3(r), H)[b % 5]))
    for k in range(8):
        b = int(r.integers(n))
        others = [q for q in range(n) if q != b]
        picked = [int(q) for q in r.permutation(others)[:int(r.integers(0, min(4, n)))]]
        mask = sum(1 << q for q in picked)
        value = sum(1 << q for q in picked if r.integers(2))
        out.append((b, mask, value, (_u3(r), X, Z, T, Y, H, _u3(r), X)[k]))
    for b in range(n):
        out.append((b, 0, 0, _u3(r)))
    half = np.diag([1, 0.5]) @ _u3(r)
    out += [(0, 0, 0, half), (n - 1, 0, 0, np.linalg.inv(half) * 0.5)]
    return out


def _reference(a, gates, n):
    a = a.copy()
    i = np.arange(1 << n)
    for b, mask, value, m in gates:
        m = np.asarray(m, np.complex128)
        lo = i[((i & mask) == value) & ((i >> b & 1) == 0)]
        hi = lo | 1 << b
        x, y = a[lo], a[hi]
        a[lo], a[hi] = m[0, 0] * x + m[0, 1] * y, m[1, 0] * x + m[1, 1] * y
    return a


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 11, 12, 13, 14, 19, 20])
def test_programs(n, scaled, dtype):
    print("programs", n, scaled, np.dtype(dtype).name, flush=True)
    sys.stdout.flush()
    r = np.random.default_rng(7 * n + scaled)
    gates = _gates(n, r)
    a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(dtype)
    ops = hq.make_ops(*zip(*gates))
    if scaled:
        t = N.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=3,
                             kernel=N.HGM_KERNEL_REG,
                             planner=N.HGM_PLAN_GREEDY | N.HGM_PLAN_FUSE | N.HGM_PLAN_PIVOT)
    else:
        t = N.default_tuning()
    plan = hq.Plan(n, ops, t, 1, dtype)
    s = hq.State(n, dtype)
    for _ in range(2):   # the second run finds the plan's tables on the device
        s.upload(a)
        plan.run(s)
        got = s.download().astype(np.complex128)
        want = _reference(a.astype(np.complex128), gates, n)
        bound = 16 * np.finfo(dtype).eps * len(gates) * 2**4 * np.linalg.norm(want)
        assert np.linalg.norm(got - want) <= bound
