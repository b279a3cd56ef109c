"""Phases under run-time conditions in the plan-compiled kernels: as many on the
same registers as lie below, at and above the size from which they are gathered
into one factor per lane, real and complex, on set and clear bits of the
thread, the register and the tile. Reference: numpy, FP64. A phase rounds an
amplitude at most 8 times (a complex product, and one in the factor): 8 eps per
phase, relative to the state's norm."""
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu


def _case(n, count, r):
    """count phases on every target, each with one or two controls of any value."""
    gates = []
    for b in range(n):
        for k in range(count):
            picked = [int(q) for q in r.permutation([q for q in range(n) if q != b])[:1 + k % 2]]
            mask = sum(1 << q for q in picked)
            value = sum(1 << q for q in picked if r.integers(2))
            gates.append((b, mask, value, np.diag([1, -1 if k % 3 == 1 else np.exp(1j * r.uniform(0, 6))])))
    return gates


def _run(n, gates, a, dtype):
    t = N.default_tuning(block_size=64, repeat_count=8, gpu_region_bits=10, gpu_coalesced_bits=3, kernel=N.HGM_KERNEL_JIT)
    plan = hq.Plan(n, hq.make_ops(*zip(*gates)), t, 1, dtype)
    assert plan.kernel == N.HGM_KERNEL_JIT
    s = hq.State(n, dtype)
    s.upload(a)
    plan.run(s)
    return s.download().astype(np.complex128)


def _factors(n, gates):
    i = np.arange(1 << n)
    f = np.ones(1 << n, np.complex128)
    for b, mask, value, m in gates:
        f[((i & mask) == value) & (i >> b & 1 == 1)] *= m[1, 1]
    return f


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [10, 11, 14])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 9])
def test_gathered_phases(count, n, dtype):
    print("phases", count, n, np.dtype(dtype).name, flush=True)
    sys.stdout.flush()
    r = np.random.default_rng(31 * n + count)
    gates = _case(n, count, r)
    a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(dtype)
    want = a.astype(np.complex128) * _factors(n, gates)
    assert np.linalg.norm(_run(n, gates, a, dtype) - want) <= 8 * np.finfo(dtype).eps * len(gates) * np.linalg.norm(want)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_an_infinity_that_no_phase_touches_stays_one(dtype):
    n = 12
    r = np.random.default_rng(3)
    gates = _case(n, 6, r)
    touched = np.zeros(1 << n, bool)
    i = np.arange(1 << n)
    for b, mask, value, _ in gates:
        touched |= ((i & mask) == value) & (i >> b & 1 == 1)
    at = int(np.flatnonzero(~touched)[-1])
    a = np.ones(1 << n, dtype)
    a[at] = np.inf
    got = _run(n, gates, a, dtype)
    assert got[at] == np.inf and np.all(np.isfinite(np.delete(got, at)))
