"""Serving requests at the limit of the server's device memory: the forms that
a request's programs can take, from the largest to the smallest.

The server's arena is sized from the programs' own sizes: a request with
compiled and interpreted passes holds both forms of its programs; where they do
not fit it runs interpreted; where its usual interpreted programs do not fit
either, compact ones. Reference: the same gates applied in FP64. An amplitude
is off by at most 4 eps per gate (a 2-term product with rounded coefficients)."""
import ctypes as C
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N
from simulador_quantico_amd import serving as S

pytestmark = pytest.mark.gpu

n = 15
STATE = 8 << n


def _u3(r):
    z, _ = np.linalg.qr(r.normal(size=(2, 2)) + 1j * r.normal(size=(2, 2)))
    return z


def _layers(depth, r):
    gates = []
    for k in range(depth):
        gates += [(b, 0, 0, _u3(r)) for b in range(n)]
        gates += [(b, 2 << b, 2 << b, np.diag([1, -1])) for b in range(k % 2, n - 1, 2)]
    return gates


def _sizes(server, gates):
    """Bytes of a request's register program, of that with its maps, of its interpreted programs and of compact ones."""
    t = N.default_tuning(**server.tuning(n))
    p = hq.Plan(n, hq.make_ops(*zip(*gates)), t, 1, np.complex64)
    assert p.kernel == N.HGM_KERNEL_REG
    rops = 104 * sum(len(p.program(i)[0]) for i in range(len(p)))
    return rops, rops + 256 * len(p.maps()) + 2056 * len(p), len(p.exec_program()[1]), len(p.exec_program(True)[1])


def _server(arena):
    return S.Server(np.complex64, hbm_budget_gib=arena / 2**30, planner_threads=1)


def _serve(server, gates):
    out = np.zeros(1 << n, np.complex64)
    rid = server.submit(n, S.ops_np(hq.make_ops(*zip(*gates))), 3, state_out=out)
    got = []
    while not got:
        got = server.poll(timeout_ms=1000)
    assert got[0]["id"] == rid
    return got[0]["status"], out


def _reference(gates):
    s = hq.State(n, np.complex128)
    s.set_basis(3)
    s.apply(hq.make_ops(*zip(*gates)))
    return s.download()


def _accepted(server, gates):
    status, out = _serve(server, gates)
    assert status == N.HGM_OK
    assert np.linalg.norm(out - _reference(gates)) <= 4 * np.finfo(np.float32).eps * len(gates)


def test_compiled_and_interpreted_passes_in_little_memory():
    r = np.random.default_rng(1)
    head = _layers(2, r)
    gates = head + _layers(300, r)
    shape = dict(ops_block=len(head))   # the first two layers are planned by themselves: one pass of theirs is compiled
    sizes = {}
    with _server(64 << 20) as big:
        big.set_tuning(n, **shape)
        assert big.precompile(n, S.ops_np(hq.make_ops(*zip(*head)))) > 0
        rops, _, usual, _ = _sizes(big, gates)
        sizes = dict(both=STATE + rops + usual, interpreted=STATE + usual)
        print("serving memory", sizes, flush=True)
        _accepted(big, gates)
    arena = sizes["interpreted"] + (64 << 10)
    assert (1 << 20) <= arena + (256 << 10) < sizes["both"]
    with _server(max(arena, 1 << 20)) as tight:
        tight.set_tuning(n, **shape)
        assert tight.precompile(n, S.ops_np(hq.make_ops(*zip(*head)))) > 0
        _accepted(tight, gates)
        _accepted(tight, head)   # all compiled, or small: as ever


def test_interpreted_passes_in_little_memory():
    """Gates on one qubit that nothing fuses: the usual programs take more than the register program and its maps, in
    whose memory the request has to fit."""
    r = np.random.default_rng(2)
    gates = [(9, 1 << 10 if k % 2 else 0, 1 << 10 if k % 2 else 0, _u3(r)) for k in range(8000)]
    with _server(64 << 20) as big:
        _, register, usual, compact = _sizes(big, gates)
        _accepted(big, gates)
    arena = STATE + register + (16 << 10)
    print("serving memory", register, usual, compact, arena, flush=True)
    sys.stdout.flush()
    assert STATE + usual > arena > STATE + compact
    with _server(arena) as tight:
        _accepted(tight, gates)
    with _server(STATE + compact // 2 + (512 << 10)) as small:   # enough for compact programs
        _accepted(small, gates[:7000])
    with _server(1 << 20) as none:                               # not even for those
        assert _serve(none, gates * 3)[0] == N.HGM_E_ARG
