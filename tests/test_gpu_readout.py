"""Whole-state reductions (probabilities of a qubit, norm, argmax) at the sizes
where the blocks' rounds change: fewer amplitudes than a block, one load per
lane, eight loads per lane, and borrowed states that are aligned to one
amplitude only. Reference: the same sums in numpy, FP64. Both sides add 2^n
non-negative terms pairwise or in short chains, so they differ by at most a
few hundred roundings of the sum: 1e-13 relative."""
import ctypes as C
import sys

import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 8, 11, 20, 21, 22, 23])
def test_reductions(n, shift, dtype):
    print("reductions", n, shift, np.dtype(dtype).name, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(100 * n + shift)
    a = (rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)).astype(dtype)
    a /= np.sqrt(np.sum(np.abs(a.astype(np.complex128)) ** 2)).astype(a.real.dtype)
    room = hq.State(n + 1, dtype)
    h = C.c_void_p()
    code = N.HGM_C64 if dtype == np.complex64 else N.HGM_C128
    at = N.lib.hgm_state_device_ptr(room._h) + shift * a.itemsize
    assert at % 16 == (8 if shift and dtype == np.complex64 else 0)
    N.check(N.lib.hgm_state_wrap(at, n, code, C.byref(h)))
    s = hq.State.__new__(hq.State)
    s.dtype, s.qubits, s._h = np.dtype(dtype), n, h
    s.upload(a)
    w = a.astype(np.complex128)
    p = w.real * w.real + w.imag * w.imag
    assert abs(s.norm2() - p.sum()) <= 1e-13 * p.sum()
    for q in {0, n // 2, n - 1}:
        halves = p.reshape(1 << q, 2, -1).sum(axis=(0, 2))
        assert np.all(np.abs(np.array(s.prob_halves(q)) - halves) <= 1e-13 * p.sum())
        assert abs(s.prob_one(q) - halves[1]) <= 1e-13 * p.sum()
    index, top = s.argmax()
    assert index == int(np.argmax(p)) and abs(top - p[index]) <= 4e-16 * top
    a[: 1 << (n - 1)] = a[1 << (n - 1):]          # every value twice: the lowest index wins
    s.upload(a)
    w = a.astype(np.complex128)
    assert s.argmax()[0] == int(np.argmax(w.real * w.real + w.imag * w.imag))
