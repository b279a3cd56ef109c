"""Batch graphs whose states share launches, a branch or a plan of any kernel
family: every state starts from amplitudes of its own and has to end where its
plan alone takes it, bit for bit (the same kernels on the same numbers)."""
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)


def _plan(n, kernel, phase, dtype, r=12):
    gates = []
    for layer in range(2):
        gates += [(b, 0, 0, H) for b in range(n)]
        gates += [(b, 2 << b, 2 << b, np.diag([1, np.exp(1j * (phase + b))])) for b in range(layer, n - 1, 2)]
    t = N.default_tuning(block_size=1 << (r - 4), repeat_count=8, gpu_region_bits=r, gpu_coalesced_bits=3, kernel=kernel)
    p = hq.Plan(n, hq.make_ops(*zip(*gates)), t, 1, dtype)
    assert p.kernel == kernel
    return p


def _check(plans, dtype):
    sizes = [p.qubits for p in plans]
    r = np.random.default_rng(len(plans))
    start = [(r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(dtype) for n in sizes]
    want = []
    for n, p, a in zip(sizes, plans, start):
        s = hq.State(n, dtype)
        s.upload(a)
        p.run(s)
        want.append(s.download())
    assert len({w.tobytes() for w in want}) == len(want)
    states = [hq.State(n, dtype) for n in sizes]
    batch = hq.Batch(states, plans)
    for replay in range(3):
        for s, a in zip(states, start):
            s.upload(a)
        batch.run()
        for k, s in enumerate(states):
            assert np.array_equal(s.download(), want[k]), (replay, k)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("kernel", [N.HGM_KERNEL_REG, N.HGM_KERNEL_LDS, N.HGM_KERNEL_JIT])
@pytest.mark.parametrize("n", [9, 12, 15])
def test_states_on_one_plan(n, kernel, dtype):
    print("one plan", n, kernel, np.dtype(dtype).name, flush=True)
    sys.stdout.flush()
    r = 12 if n >= 12 else 8
    p = _plan(n, kernel, 0.3, dtype, r)
    group, _ = hq.Batch.layout([p] * 5)
    assert len(set(group)) == (5 if kernel == N.HGM_KERNEL_LDS else 1)
    _check([p] * 5, dtype)


def test_more_groups_than_branches():
    plans = [_plan(9, (N.HGM_KERNEL_REG, N.HGM_KERNEL_LDS)[k % 2], 0.05 * (k // 2 + 1), np.complex64, 8) for k in range(140)]
    group, branch = hq.Batch.layout(plans)
    assert len(set(group)) == 140 and len(set(branch)) == 64
    print("groups", len(set(group)), "branches", len(set(branch)), flush=True)
    _check(plans, np.complex64)


def test_groups_of_every_family_side_by_side():
    reg, jit = _plan(14, N.HGM_KERNEL_REG, 0.3, np.complex64), _plan(13, N.HGM_KERNEL_JIT, 0.4, np.complex64)
    lds, twin = _plan(13, N.HGM_KERNEL_LDS, 0.5, np.complex64), _plan(14, N.HGM_KERNEL_REG, 0.3, np.complex64)
    plans = [reg, lds, jit, twin, lds, reg, jit]
    group, _ = hq.Batch.layout(plans)
    assert group[0] == group[3] == group[5] and group[2] == group[6] and group[1] != group[4]
    print("families", group, flush=True)
    _check(plans, np.complex64)
