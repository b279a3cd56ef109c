"""What hgm_state_apply_noalloc takes: any plan whose own table fits the 8 MiB
workspace, whatever other forms of its program would need."""
import ctypes as C
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)
X = np.array([[0, 1], [1, 0]])
WORKSPACE = 8 << 20


def _run(fn, n, ops, tun, a):
    s = hq.State(n, a.dtype)
    s.upload(a)
    st = N.Stats()
    rc = fn(s._h, ops, len(ops), C.byref(tun), 1, C.byref(st))
    return rc, s.download()


def _tuning():
    return N.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=3, kernel=N.HGM_KERNEL_REG,
                            ops_block=1 << 30)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_a_plan_is_measured_by_the_table_that_it_sends(dtype):
    """90000 gates, most of them X, which cost no record: the inspected register program is above 8 MiB, the table that is
    sent far below."""
    n = 12
    ops = hq.make_ops(*zip(*[(k % n, 0, 0, H if k % 50 == 0 else X) for k in range(90000)]))
    plan = hq.Plan(n, ops, _tuning(), 1, dtype)
    assert sum(len(plan.program(i)[0]) for i in range(len(plan))) * 104 > WORKSPACE > 4 * len(plan.exec_program()[1])
    print("noalloc table", np.dtype(dtype).name, len(plan.exec_program()[1]), flush=True)
    sys.stdout.flush()
    r = np.random.default_rng(1)
    a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(dtype)
    rc, want = _run(N.lib.hgm_state_apply, n, ops, _tuning(), a)
    assert rc == N.HGM_OK
    rc, got = _run(N.lib.hgm_state_apply_noalloc, n, ops, _tuning(), a)
    assert rc == N.HGM_OK, N.lib.hgm_last_error()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_a_plan_whose_usual_table_does_not_fit_runs_compact(dtype):
    """Gates on one qubit, and in FP64 phases between them: 8 MiB hold the register program but not the usual table.
    Reference: the gates' product in FP64. A gate rounds an amplitude by a 2-term complex product, at most 4 eps."""
    n, q, count = 12, 5, 60000
    r = np.random.default_rng(2)
    few = []
    for k in range(16):
        z, _ = np.linalg.qr(r.normal(size=(2, 2)) + 1j * r.normal(size=(2, 2)))
        few.append(z if dtype == np.complex64 or k % 2 else np.diag(np.exp(1j * r.uniform(0, 6, 2))))
    picked = [few[int(k)] if dtype == np.complex64 else few[2 * int(k // 2) + i % 2] for i, k in enumerate(r.integers(0, 16, count))]
    if dtype == np.complex128:
        picked = picked[:52000]
    ops = hq.make_ops([q] * len(picked), [0] * len(picked), [0] * len(picked), [m.reshape(4) for m in picked])
    plan = hq.Plan(n, ops, _tuning(), 1, dtype)
    assert len(plan.exec_program()[1]) > WORKSPACE >= sum(len(plan.program(i)[0]) for i in range(len(plan))) * 104 + 65536
    print("noalloc compact", np.dtype(dtype).name, len(plan.exec_program()[1]), len(plan.exec_program(True)[1]), flush=True)
    sys.stdout.flush()
    u = np.eye(2, dtype=np.clongdouble)
    for m in picked:
        u = m.astype(np.clongdouble) @ u
    a = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)).astype(dtype)
    want = np.einsum("ij,ajb->aib", u.astype(np.complex128), a.astype(np.complex128).reshape(-1, 2, 1 << q)).reshape(-1)
    rc, got = _run(N.lib.hgm_state_apply_noalloc, n, ops, _tuning(), a)
    assert rc == N.HGM_OK, N.lib.hgm_last_error()
    assert np.linalg.norm(got - want) <= 4 * np.finfo(dtype).eps * len(picked) * np.linalg.norm(want)
