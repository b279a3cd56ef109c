"""The programs that the interpreted register kernels run (csrc/program.hpp),
executed by a numpy model of the kernel's semantics, must reproduce the oracle
on every launch shape; and their coefficients must be as exact as the kernels
rely on.

The model follows k_pass_reg: a launch gives every tile of 2^r amplitudes to a
workgroup, thread t holds A of them in registers; records act on registers, and
a remap moves the tile through LDS. What a barrier-free remap and a single
barrier per remap rely on is checked with it."""
import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N
from simulador_quantico_amd.dgm import XMAP_DTYPE, XPASS_DTYPE, xop_dtype
from tests.test_oracle import _random_gate_list, oracle_run_gates

(X_DENSE, X_DENSE_REAL, X_ROT, X_ROTS, X_SWAP, X_DENSE_LANE, X_REAL_LANE, X_DENSE_MASK, X_REAL_MASK, X_PHASE, X_VEC,
 X_VEC_REAL, X_REMAP) = range(13)
X_FIRST, X_LAST, X_REAL = 1, 2, 4
X_PAT_CLEAR, X_PAT_MASK = 32, 255
REAL = {np.complex64: np.float32, np.complex128: np.float64}


def _records(prog, at, dtype):
    head = prog[at:at + 512].view(XPASS_DTYPE)[0]
    op = xop_dtype(REAL[dtype])
    n = int(head["n_ops"])
    ops = prog[at + 512:at + 512 + (n + 1) * op.itemsize].view(op)
    assert int(ops[n]["kind"]) == 0 and not ops[n]["m"].any()   # the record that the kernel loads ahead
    return head, ops[:n], prog[at + int(head["table"]):]


def _deposit(v, runs, n):
    x = np.zeros_like(v)
    for r in runs[:n]:
        x |= ((v >> np.uint64(r["from"])) & np.uint64(r["mask"])) << np.uint64(r["to"])
    return x


def _bits(k, bits):
    x = np.zeros(len(k), np.uint64)
    for i, b in enumerate(bits):
        x ^= np.where(k >> i & 1 == 1, np.uint64(b), np.uint64(0))
    return x


def _slots(m, B, A, fold):
    """LDS slot of (thread, register)."""
    a, x = A.bit_length() - 1, np.arange(B, dtype=np.int64)
    for i in range(a):
        x = x + (x & ~int(m["low"][i]))
    mask = (1 << fold) - 1
    x ^= (x >> fold & mask) ^ (x >> 2 * fold & mask) ^ (x >> 3 * fold & mask)
    return x[:, None] ^ _bits(np.arange(A), m["sw"][:a]).astype(np.int64)[None, :]


def _phase_factor(o):
    return np.frombuffer(o["m"].tobytes()[:16], np.float64)


def _selected(o, A):
    k, pat = np.arange(A), int(o["pat"])
    if pat == X_PAT_MASK:
        return (int(o["pmask"]) >> k & 1) == 1
    if pat >= X_PAT_CLEAR:
        return (k >> (pat - X_PAT_CLEAR) & 1) == 0
    return (k & pat) == pat


def emulate(plan, n, psi, dtype, compact=False):
    (r, A, B, sync), prog, launches = plan.exec_program(compact)
    a_bits, fold = A.bit_length() - 1, 5 if dtype == np.complex64 else 4
    k, t = np.arange(A), np.arange(B, dtype=np.uint64)
    psi = psi.astype(np.complex128).copy()
    for at, stages in launches:
        head, ops, table = _records(prog, int(at), dtype)
        assert 1 + sum(int(o["kind"]) == X_REMAP for o in ops) == stages
        base = _deposit(np.arange(1 << (n - r), dtype=np.uint64), head["base"], int(head["n_base"]))
        load = _deposit(t, head["load"], int(head["n_load"]))
        store = _deposit(t, head["store"], int(head["n_store"])) ^ head["sflip"]
        idx = (base[:, None, None] | load[None, :, None]) + _bits(k, head["lbit"][:a_bits])[None, None, :]
        out = (base[:, None, None] | store[None, :, None]) + (_bits(k, head["sbit"][:a_bits]) ^ head["rflip"])[None, None, :]
        for i in (idx, out):   # every amplitude once
            assert np.array_equal(np.sort(i.reshape(-1)), np.arange(1 << n, dtype=np.uint64))
        a = psi[idx.astype(np.int64)]
        cur = head["first"]
        group = None
        for o in ops:
            kind = int(o["kind"])
            if kind == X_REMAP:
                to = np.frombuffer(o["m"].tobytes()[:32], XMAP_DTYPE)[0]
                w, rd = _slots(cur, B, A, fold), _slots(to, B, A, fold)
                assert np.array_equal(np.sort(w.reshape(-1)), np.arange(1 << r))
                assert np.array_equal(np.sort(rd.reshape(-1)), np.arange(1 << r))
                if not sync:   # a tile lies within a wave: readers find their own wave's slots
                    wave = np.zeros(1 << r, np.int64)
                    wave[w] = (np.arange(B) // 64)[:, None]
                    assert (wave[rd] == (np.arange(B) // 64)[:, None]).all()
                lds = np.zeros((a.shape[0], 1 << r), complex)
                lds[:, w] = a
                a = lds[:, rd]
                cur = to
                continue
            tile = (base & o["gmask"]) == o["gval"]
            lane = (t & np.uint64(o["tmask"])) == np.uint64(o["tval"])
            if kind == X_PHASE:
                f = _phase_factor(o)
                g = np.where(tile[:, None] & lane[None, :], f[0] + 1j * f[1], 1)
                if int(o["flags"]) & X_FIRST:
                    assert group is None
                    group = np.ones_like(g)
                assert not int(o["flags"]) & X_REAL or f[1] == 0
                group = group * g
                if int(o["flags"]) & X_LAST:
                    a[:, :, _selected(o, A)] *= group[:, :, None]
                    group = None
                continue
            assert group is None
            m = o["m"].astype(np.float64)
            if kind in (X_VEC, X_VEC_REAL):
                f = table.view(REAL[dtype])[int(o["pmask"]):][:2 * A].astype(np.float64)
                a *= f[:A] if kind == X_VEC_REAL else f[0::2] + 1j * f[1::2]
                continue
            for b in range(min(4, a_bits)) if kind == X_ROTS else [int(o["bit"])]:
                lo = k[(k >> b & 1) == 0]
                x, y = a[:, :, lo].copy(), a[:, :, lo | 1 << b].copy()
                where = tile[:, None, None] & np.ones((1, B, len(lo)), bool)
                if kind == X_ROTS:
                    p, q = x + m[2 * b] * y, y + m[2 * b + 1] * x
                elif kind == X_ROT:
                    t0, t1 = (m[0], m[1]) if dtype == np.complex64 else (m[0] + 1j * m[1], m[2] + 1j * m[3])
                    p, q = x + t0 * y, y + t1 * x
                elif kind == X_SWAP:
                    p, q, where = y, x, where & lane[None, :, None]
                else:
                    c = m[0::2] + 1j * m[1::2]
                    if kind in (X_DENSE_REAL, X_REAL_LANE, X_REAL_MASK):
                        assert not c.imag.any()
                    p, q = c[0] * x + c[1] * y, c[2] * x + c[3] * y
                    if kind not in (X_DENSE, X_DENSE_REAL):
                        where = where & lane[None, :, None]
                    if kind in (X_DENSE_MASK, X_REAL_MASK):
                        where = where & (int(o["pmask"]) >> lo & 1 == 1)[None, None, :]
                a[:, :, lo] = np.where(where, p, x)
                a[:, :, lo | 1 << b] = np.where(where, q, y)
        psi[out.astype(np.int64)] = a
    return psi


def _compare(n, gates, tuning, dtype, r):
    """Each gate is a few products with coefficients rounded to the amplitude type: 16 eps per gate, as its kernel has."""
    t, cm, cv, mats = gates
    plan = hq.Plan(n, hq.make_ops(t, cm, cv, mats), tuning, 1, dtype)
    assert plan.kernel == N.HGM_KERNEL_REG
    psi = r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)
    psi /= np.linalg.norm(psi)
    want = oracle_run_gates(n, t, cm, cv, mats, state=psi)
    off = np.linalg.norm(emulate(plan, n, psi, dtype) - want)
    assert off <= 16 * np.finfo(dtype).eps * len(t), off
    return plan


def _tunings(n, dtype):
    """Every tile shape the register kernels accept at n qubits."""
    for r in range(1, 15 if dtype == np.complex64 else 14):
        for rl in range(0, min(5, r)):
            B, R = 1 << (r - 1 - rl), 1 << rl
            for c in range(0, r + 1):
                t = N.default_tuning(block_size=B, repeat_count=R, gpu_region_bits=r, gpu_coalesced_bits=c, kernel=N.HGM_KERNEL_REG)
                yield t


PLANNERS = (N.HGM_PLAN_GREEDY, N.HGM_PLAN_GREEDY | N.HGM_PLAN_FUSE | N.HGM_PLAN_PIVOT, N.HGM_PLAN_GREEDY | N.HGM_PLAN_ROTATE)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", range(1, 15))
def test_programs_match_the_oracle_on_every_shape(n, dtype):
    """All shapes are planned and their launch limits checked; a few of each size are run."""
    r = np.random.default_rng(100 * n + (dtype == np.complex64))
    accepted = []
    few = hq.make_ops(*_random_gate_list(r, n, 4)) if n > 1 else hq.make_ops([0], [0], [0], [np.eye(2)[::-1].reshape(4)])
    size = np.dtype(dtype).itemsize
    for t in _tunings(n, dtype):
        try:
            p = hq.Plan(n, few, t, 1, dtype)
        except N.HGMError:
            continue
        accepted.append(t)
        (tile, A, B, sync), _, launches = p.exec_program()
        most = {4: 1024, 8: 1024, 2: 1024, 16: 1024 if size == 8 else 512, 32: 512 if size == 8 else 256}[A]
        assert A * B == 1 << tile and B <= most and tile <= n and size << tile <= 160 * 1024 - 1024
        assert B >= 64 or tile == n
        assert sync or B <= 64
    assert accepted
    for i in r.permutation(len(accepted))[:6 if n > 11 else 12]:
        t = accepted[int(i)]
        t.planner = PLANNERS[int(i) % len(PLANNERS)]
        print("shape", n, np.dtype(dtype).name, t.as_dict() if hasattr(t, "as_dict") else i)
        _compare(n, _random_gate_list(r, n, 60), t, dtype, r)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [2, 8, 11, 13, 14])
def test_programs_of_the_default_tuning(n, dtype):
    r = np.random.default_rng(n)
    _compare(n, _random_gate_list(r, n, 120), N.default_tuning(kernel=N.HGM_KERNEL_REG), dtype, r)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_a_whole_state_plan_of_several_launches(dtype):
    """One workgroup runs a small state's passes in one launch, up to 2^15 gates: this plan has two."""
    n = 4
    r = np.random.default_rng(9)
    t, cm, cv, mats = _random_gate_list(r, n, 150)
    times = 230
    tuning = N.default_tuning(block_size=2, repeat_count=2, gpu_region_bits=3, gpu_coalesced_bits=1, kernel=N.HGM_KERNEL_REG)
    plan = _compare(n, (t * times, cm * times, cv * times, mats * times), tuning, dtype, r)
    assert len(plan.exec_program()[2]) == 2 < len(plan)


def test_fp64_programs_hold_whole_gates():
    """In FP64 a split into rotations and phases rounds more than the gate itself: every record holds the entries of one
    gate, bit for bit, and no rotation but a row-scaled gate's, whose other entries are exact ones."""
    n = 13
    r = np.random.default_rng(4)
    t, cm, cv, mats = _random_gate_list(r, n, 150)
    entries = {complex(z) for m in mats for z in m} | {1, 0}
    tuning = N.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=3, kernel=N.HGM_KERNEL_REG)
    _, prog, launches = hq.Plan(n, hq.make_ops(t, cm, cv, mats), tuning, 1, np.complex128).exec_program()
    seen = 0
    for at, _ in launches:
        for o in _records(prog, int(at), np.complex128)[1]:
            kind = int(o["kind"])
            assert kind not in (X_ROT, X_ROTS)
            if kind not in (X_VEC, X_VEC_REAL, X_REMAP, X_SWAP, X_PHASE):
                assert {complex(x, y) for x, y in o["m"].reshape(4, 2)} <= entries
                seen += 1
    assert seen > 20
    tuning.planner = N.HGM_PLAN_GREEDY | N.HGM_PLAN_PIVOT
    ops = (N.Op * (2 * len(t) + n + 1))()
    import ctypes as C
    count = C.c_int64()
    N.check(N.lib.hgm_pivot_rows(n, hq.make_ops(t, cm, cv, mats), len(t), ops, len(ops), C.byref(count)))
    entries = {complex(o.m[2 * i], o.m[2 * i + 1]) for o in ops[:count.value] for i in range(4)} | {1, 0}
    _, prog, launches = hq.Plan(n, hq.make_ops(t, cm, cv, mats), tuning, 1, np.complex128).exec_program()
    kinds = []
    for at, _ in launches:
        for o in _records(prog, int(at), np.complex128)[1]:
            kinds.append(int(o["kind"]))
            if kinds[-1] == X_ROT:
                assert {complex(o["m"][0], o["m"][1]), complex(o["m"][2], o["m"][3])} <= entries
    assert X_ROT in kinds and X_ROTS not in kinds


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_conditional_phases_are_not_rounded(dtype):
    """The factor of a group of phases is multiplied up in FP64: the records hold the gates' own doubles."""
    n = 13
    r = np.random.default_rng(5)
    z = np.exp(1j * r.uniform(0, 6, 40))
    t = [int(b) for b in r.integers(0, 4, 40)]
    cm = [1 << int(b) for b in r.integers(4, 8, 40)]
    _, prog, launches = hq.Plan(n, hq.make_ops(t, cm, cm, [np.array([1, 0, 0, x]) for x in z]),
                                N.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=3,
                                                 kernel=N.HGM_KERNEL_REG), 1, dtype).exec_program()
    single = {(b, m): [x for x, c, d in zip(z, t, cm) if (c, d) == (b, m)] for b, m in zip(t, cm)}
    single = {v[0] for v in single.values() if len(v) == 1}
    found = {complex(*_phase_factor(o)) for at, _ in launches for o in _records(prog, int(at), dtype)[1] if int(o["kind"]) == X_PHASE}
    assert single and single <= found


def _register_bytes(plan):
    """The register program, its maps and its pass tables."""
    rops = sum(len(plan.program(i)[0]) for i in range(len(plan)))
    return 104 * rops + 256 * len(plan.maps()) + 2056 * len(plan)


def _u3(r):
    z, _ = np.linalg.qr(r.normal(size=(2, 2)) + 1j * r.normal(size=(2, 2)))
    return z.reshape(4)


def _families(n, r):
    """Gate lists whose usual programs are large: little that merges, much that needs a factor per register."""
    k = 300
    one = [int(n // 2)] * k
    yield "one qubit", (one, [0] * k, [0] * k, [_u3(r) for _ in range(k)])
    rz = [np.array([np.exp(-1j * x), 0, 0, np.exp(1j * x)]) for x in r.uniform(0, 3, k)]
    yield "turns", (one, [0] * k, [0] * k, [rz[i] if i % 2 else _u3(r) for i in range(k)])
    other = 1 << (n // 2 + 1)
    yield "controls", (one, [0 if i % 2 else other for i in range(k)], [0 if i % 2 else other * (i // 2 % 2) for i in range(k)],
                       [_u3(r) if i % 2 else rz[i] for i in range(k)])
    anti = [np.array([0, np.exp(1j * x), np.exp(-1j * x), 0]) for x in r.uniform(0, 3, k)]
    yield "exchanges", (one, [0] * k, [0] * k, anti)
    yield "any", _random_gate_list(r, n, k)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [4, 9, 13])
def test_compact_programs_take_no_more_than_the_register_program(n, dtype):
    r = np.random.default_rng(n)
    larger = 0
    for name, (t, cm, cv, mats) in _families(n, r):
        for amps in (2, 4, 16):
            for ops_block in (1, 40, 1 << 30):
                bits = min(n, 11) if n > 4 else 4
                tuning = N.default_tuning(block_size=max(1, (1 << bits) // amps), repeat_count=amps // 2, gpu_region_bits=bits,
                                          gpu_coalesced_bits=min(3, bits - 1), kernel=N.HGM_KERNEL_REG, ops_block=ops_block)
                plan = hq.Plan(n, hq.make_ops(t, cm, cv, mats), tuning, 1, dtype)
                limit = _register_bytes(plan)
                assert len(plan.exec_program(True)[1]) <= limit, (name, amps, ops_block)
                larger += len(plan.exec_program()[1]) > limit
        psi = r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)
        psi /= np.linalg.norm(psi)
        off = np.linalg.norm(emulate(plan, n, psi, dtype, True) - oracle_run_gates(n, t, cm, cv, mats, state=psi))
        assert off <= 16 * np.finfo(dtype).eps * len(t), (name, off)
    assert larger   # what the compact form is for
