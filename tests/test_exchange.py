"""The LDS exchanges of the generated pass kernels, executed on the CPU from the
generated source: every slot in bounds, no slot shared by two threads between
barriers unless all of them read it, and every element where the phase map of the
next phase has it."""
import ctypes as C
import re

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

_LINE = re.compile(r"const unsigned (\w+) = (.*);|lds\[(f\d+) \+ (\d+)u\] = a(\d+)(\.[xy])?;"
                   r"|a(\d+)(\.[xy])? = lds\[(f\d+) \+ (\d+)u\];|(__syncthreads)\(\);")


def _index(m, B, A):
    """Tile index of (thread, register): maps hold it XOR-swizzled."""
    t, k = np.arange(B)[:, None], np.arange(A)[None, :]
    x = m["thr"].reshape(2, 32)[0][t & 31] ^ m["thr"].reshape(2, 32)[1][t >> 5] ^ m["reg"].ravel()[k]
    return (x ^ (x >> 4 & 15) ^ (x >> 8 & 15) ^ (x >> 12 & 15)).astype(np.int64)


def _sequences(plan):
    maps = plan.maps()
    for i in range(len(plan)):
        _, first, last, _ = plan.program(i)
        yield i, [maps[m] for m in range(first, last + 1)]


def _run(src, seq, B, A, entries, split):
    """Checks one kernel's exchanges against a pass's maps: (slots in bounds and
    free of races, elements where the maps have them, exchanges done)."""
    comps = [".x", ".y"] if split else [None]
    regs = {c: _index(seq[0], B, A) for c in comps}
    lds = np.full(entries, -1, np.int64)
    env = {"t": np.arange(B)}
    writer, reader = np.full(entries, -1), np.full(entries, -1)
    safe = True
    reads = {c: 0 for c in comps}
    done = 0
    for mt in _LINE.finditer(src):
        if mt[1]:
            if re.fullmatch(r"[xf]\d+", mt[1]):
                expr = re.sub(r"\(unsigned( long long)?\)|(?<=[0-9a-f])(ull|u)\b", "", mt[2])
                env[mt[1]] = np.asarray(eval(expr, {}, env)) + np.zeros(B, np.int64)
        elif mt[3]:
            at = (env[mt[3]] + int(mt[4])).astype(np.int64)
            safe &= at.max() < entries and len(set(at)) == B
            if not safe:
                return False, False, done
            other = (reader[at] >= 0) & (reader[at] != np.arange(B)) | (writer[at] >= 0) & (writer[at] != np.arange(B))
            safe &= not other.any()
            writer[at] = np.arange(B)
            lds[at] = regs[mt[6]][:, int(mt[5])]
        elif mt[7]:
            c, at = mt[8], (env[mt[9]] + int(mt[10])).astype(np.int64)
            safe &= at.max() < entries
            if not safe:
                return False, False, done
            safe &= not ((writer[at] >= 0) & (writer[at] != np.arange(B))).any()
            reader[at] = np.arange(B)
            regs[c] = regs[c].copy()
            regs[c][:, int(mt[7])] = lds[at]
            reads[c] += 1
            if all(r == A * (done + 1) for r in reads.values()):
                done += 1
                if done >= len(seq):
                    return safe, False, done
                if any((regs[x] != _index(seq[done], B, A)).any() for x in comps):
                    return safe, False, done
        elif mt[11]:
            writer[:], reader[:] = -1, -1
    return safe, done == len(seq) - 1, done


_SHAPES = [(12, 64, 1, 7, 3), (13, 64, 4, 9, 3), (15, 256, 8, 12, 4), (15, 512, 8, 13, 4), (15, 1024, 4, 13, 4),
           (16, 1024, 8, 14, 4)]


# 1024 threads of 16 complex128 amplitudes are beyond the register kernel's limits
@pytest.mark.parametrize("n,B,R,r,c,dtype", [(*s, d) for s in _SHAPES for d in (np.complex64, np.complex128)
                                             if (s[1], s[2], d) != (1024, 8, np.complex128)])
def test_exchanges_permute_in_place(n, B, R, r, c, dtype):
    d = hq.DGM()
    d.setFunction(hq.RandomLayers(n, 4, 7, d))
    A = 2 * R
    last = (1 << r) - 1
    total = 0
    for kernel in (N.HGM_KERNEL_JIT, N.HGM_KERNEL_REG):
        lo, hi = (5, 9) if kernel == N.HGM_KERNEL_REG and dtype == np.complex64 else (4, 8)   # the padding
        entries = last + (last >> lo) + (last >> hi) + 1
        split = entries * np.dtype(dtype).itemsize > 32 * 1024
        t = N.default_tuning(block_size=B, repeat_count=R, gpu_region_bits=r, gpu_coalesced_bits=c, kernel=kernel,
                             planner=N.HGM_PLAN_GREEDY | N.HGM_PLAN_FUSE, ops_block=1 << 30)
        plan = hq.Plan(n, d.ops(), t, 1, dtype)
        seqs = list(_sequences(plan))
        if kernel == N.HGM_KERNEL_JIT:   # equal passes share a kernel: each kernel fits one pass at least
            for src in plan.jit_source().split("__global__")[1:]:
                got = [_run(src, s, B, A, entries, split) for _, s in seqs]
                assert any(safe and ok for safe, ok, _ in got)
                total += max(done for safe, ok, done in got if safe and ok)
        else:
            for i, s in seqs:
                ln = C.c_size_t()
                N.check(N.lib.hgm_plan_serving_source(plan._h, i, None, 0, C.byref(ln)))
                b = C.create_string_buffer(ln.value + 1)
                N.check(N.lib.hgm_plan_serving_source(plan._h, i, b, ln.value + 1, C.byref(ln)))
                safe, ok, done = _run(b.value.decode().split("__global__")[1], s, B, A, entries, split)
                assert safe and ok
                total += done
    assert total > 0
