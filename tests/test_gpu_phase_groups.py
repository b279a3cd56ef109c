"""Phases under run-time conditions in the interpreted kernels, which multiply
all phases of a group into one factor per lane: in FP32 the factor has to be as
exact as one phase, however many phases went into it.

All phases here test thread bits and tile numbers only, so they are one group.
Bound, with u = 2^-24: the factor is a complex number of modulus 1 that is
rounded to FP32 once, per component (at most u), and a complex product of FP32
numbers is off by at most sqrt(5) u of its modulus; what the factor collects in
64 bits on the way is below 2^-40. Together 3.24 u, and 3.5 u is allowed. A
factor that is multiplied up in FP32 is off by several u more from 60 phases."""
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu

THREAD_BITS = 8   # of a tile of 2^12 amplitudes at 16 per thread: the lower ones, where no gate asks for others


def _tuning():
    return N.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=4, kernel=N.HGM_KERNEL_REG)


def _phases(n, count, r):
    """Controlled phases of distinct conditions, none with a control that has to be 0."""
    seen, gates = set(), []
    tile_bits = list(range(12, n))
    while len(gates) < count:
        picked = [int(q) for q in r.permutation(THREAD_BITS)[:2 + (len(gates) % 3 > 0)]]
        if tile_bits and len(gates) % 4 == 0:
            picked[-1] = int(r.choice(tile_bits))
        mask = sum(1 << q for q in picked)
        if mask in seen:
            continue
        seen.add(mask)
        gates.append((picked[0], mask & ~(1 << picked[0]), mask & ~(1 << picked[0]),
                      np.diag([1, np.exp(1j * r.uniform(0, 2 * np.pi))])))
    return gates


def _factors(n, gates):
    i = np.arange(1 << n)
    f = np.ones(1 << n, np.clongdouble)
    for b, mask, _, m in gates:
        on = mask | 1 << b
        f[(i & on) == on] *= np.clongdouble(m[1, 1])
    return f


@pytest.mark.parametrize("n", [12, 14])
@pytest.mark.parametrize("count", [1, 2, 5, 60])
def test_a_factor_of_many_phases_is_as_exact_as_one(count, n):
    print("phase groups", count, n, flush=True)
    sys.stdout.flush()
    for seed in range(4):
        r = np.random.default_rng(1000 * n + 10 * count + seed)
        gates = _phases(n, count, r)
        plan = hq.Plan(n, hq.make_ops(*zip(*gates)), _tuning(), 1, np.complex64)
        assert plan.kernel == N.HGM_KERNEL_REG and len(plan) == 1
        a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(np.complex64)
        s = hq.State(n, np.complex64)
        s.upload(a)
        plan.run(s)
        want = a.astype(np.clongdouble) * _factors(n, gates)
        off = np.abs(s.download().astype(np.clongdouble) - want) / np.abs(a)
        assert float(off.max()) <= 3.5 * 2.0**-24, float(off.max()) * 2**24


@pytest.mark.parametrize("n", [12, 14])
@pytest.mark.parametrize("count", [5, 60])
def test_the_compiled_kernels_factor_is_as_exact(count, n):
    """The plan-compiled kernels gather such phases too (from 3 on), into an FP64 factor: the same bound."""
    print("compiled phase groups", count, n, flush=True)
    sys.stdout.flush()
    t = _tuning()
    t.kernel = N.HGM_KERNEL_JIT
    for seed in range(2):
        r = np.random.default_rng(1000 * n + 10 * count + seed)
        gates = _phases(n, count, r)
        plan = hq.Plan(n, hq.make_ops(*zip(*gates)), t, 1, np.complex64)
        assert plan.kernel == N.HGM_KERNEL_JIT and len(plan) == 1
        a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(np.complex64)
        s = hq.State(n, np.complex64)
        s.upload(a)
        plan.run(s)
        want = a.astype(np.clongdouble) * _factors(n, gates)
        off = np.abs(s.download().astype(np.clongdouble) - want) / np.abs(a)
        assert float(off.max()) <= 3.5 * 2.0**-24, float(off.max()) * 2**24


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("real", [False, True])
def test_an_infinity_in_a_tile_that_no_phase_holds_in_stays_one(real, dtype):
    """Two phases of one group, each held in the tiles where its own state bit above the tile is set: one complex, the
    other real or complex. An infinity stays one in the tiles where neither holds and where only a real one does; the
    rest of the state has to be finite there."""
    n = 14
    print("infinity", real, np.dtype(dtype).name, flush=True)
    sys.stdout.flush()
    gates = [(0, 1 << 12, 1 << 12, np.diag([1, -1 if real else 1j])), (1, 1 << 13, 1 << 13, np.diag([1, np.exp(0.7j)]))]
    a = np.ones(1 << n, dtype)
    a[0b00 << 12 | 77] = np.inf
    if real:
        a[0b01 << 12 | 77] = np.inf
    plan = hq.Plan(n, hq.make_ops(*zip(*gates)), _tuning(), 1, dtype)
    s = hq.State(n, dtype)
    s.upload(a)
    plan.run(s)
    got = s.download()
    assert got[77] == np.inf
    if real:
        assert got[1 << 12 | 77] == -np.inf
    assert np.isfinite(got[np.isfinite(a)]).all()
