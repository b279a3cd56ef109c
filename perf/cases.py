"""Performance cases of the GPU path: what a program that uses this package has it do.

A case is a dict of plain values. "kind" names the entry point:

  plan      a resident state evolved by a kept Plan (Plan.run)
  apply     a gate list applied to a resident state in one call (State.apply)
  execute   the executor's drop-in path: DGM.execute on a host state
  readout   measurement of a resident state: both probabilities of a qubit,
            collapse, the most likely index and the norm
  batch     a fixed set of resident states of uneven sizes (Batch.run)
  serve     independent requests through the serving engine (Server)

Resident states live in torch tensors that the library borrows, so outputs are
the states' own buffers. Every circuit is a function of the case; amplitudes
and request parameters are drawn from the seed.
"""
import ctypes as C
import math

import numpy as np
import torch

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N
from simulador_quantico_amd import serving as S

NP = {"c128": np.complex128, "c64": np.complex64}
TORCH = {"c128": torch.complex128, "c64": torch.complex64}
CODE = {"c128": N.HGM_C128, "c64": N.HGM_C64}


def listed():
    return [
        # the benchmark's circuit at its full size: a 16 GiB state, compiled kernels, a plan kept over many runs
        dict(name="random30-f64", kind="plan", circuit="random", qubits=30, depth=20, dtype="c128", tuning="compiled"),
        # the same in the reference's precision: long evolutions of FP32 states
        dict(name="random30-f32", kind="plan", circuit="random", qubits=30, depth=20, dtype="c64", tuning="compiled"),
        # a search run to its end: thousands of short passes over a state that fits the last-level cache
        dict(name="grover22-f64", kind="plan", circuit="grover", qubits=22, depth=1608, dtype="c128", tuning="compiled"),
        # arithmetic by Fourier transforms: few passes, almost all gates controlled phases
        dict(name="adder29-f64", kind="plan", circuit="adder", qubits=29, depth=1, dtype="c128", tuning="compiled"),
        # parametrised circuits change at every evaluation, so they run on the interpreted kernels, where nothing is compiled
        dict(name="random27-f32-interp", kind="plan", circuit="random", qubits=27, depth=10, dtype="c64", tuning="tile"),
        # one call with the library's default tuning, as a caller of the reference has it
        dict(name="random25-f32-default", kind="apply", circuit="random", qubits=25, depth=6, dtype="c64", tuning="default"),
        # the smallest calls: a transform of a few qubits, where latency counts
        dict(name="qft11-f64-default", kind="apply", circuit="qft", qubits=11, depth=1, dtype="c128", tuning="default"),
        # the reference's general program: three Hadamard layers on a host state, copied in and out
        dict(name="hadamard24-f32-host", kind="execute", circuit="hadamard", qubits=24, depth=3, dtype="c64", tuning="default"),
        # measurement of a large state
        dict(name="readout29-f32", kind="readout", qubits=29, qubit=3, dtype="c64"),
        # many small circuits of a fixed set, run again and again as one graph
        dict(name="batch64-f32", kind="batch", states=64, qmin=12, qmax=19, depth=8, dtype="c64"),
        # a burst of small and mid-size requests on the interpreted kernels
        dict(name="serve-mix64", kind="serve", requests=64, qmin=10, qmax=16, iterations=16, depth=10, compiled=False),
        # a burst of large requests of one shape, whose kernels were compiled before
        dict(name="serve-grover23", kind="serve", requests=12, qmin=22, qmax=23, iterations=12, depth=0, compiled=True),
    ]


def draw(rng):
    kind = rng.choice(("plan", "plan", "plan", "plan", "apply", "apply", "execute", "readout", "batch", "serve"))
    dtype = rng.choice(("c128", "c64"))
    if kind in ("plan", "apply", "execute"):
        circuit = rng.choice(("random", "grover", "adder", "hadamard", "qft"))
        tuning = rng.choice(("compiled", "tile")) if kind == "plan" else "default" if kind == "execute" else rng.choice(("default", "tile"))
        lo, hi = {"plan": (16, 27 if tuning == "tile" else 29), "apply": (5, 24), "execute": (10, 24)}[kind]
        depth = {"random": rng.randint(2, 12), "grover": rng.randint(1, 48), "hadamard": rng.randint(1, 3)}.get(circuit, 1)
        qubits = rng.randint(lo, hi)
        if circuit == "adder":
            qubits |= 1
        if circuit == "grover" and qubits > 24:
            depth = 1 + depth // 8
        return dict(kind=kind, circuit=circuit, qubits=qubits, depth=depth, dtype=dtype, tuning=tuning)
    if kind == "readout":
        qubits = rng.randint(10, 29)
        return dict(kind=kind, qubits=qubits, qubit=rng.randrange(qubits), dtype=dtype)
    if kind == "batch":
        qmin = rng.randint(8, 14)
        return dict(kind=kind, states=rng.randint(6, 72), qmin=qmin, qmax=qmin + rng.randint(1, 5), depth=rng.randint(1, 12), dtype=dtype)
    if rng.random() < 0.3:
        qmin = rng.randint(20, 23)
        return dict(kind=kind, requests=rng.randint(4, 16), qmin=qmin, qmax=qmin + 1, iterations=rng.randint(2, 16), depth=0, compiled=True)
    qmin = rng.randint(10, 13)
    return dict(kind=kind, requests=rng.randint(8, 96), qmin=qmin, qmax=qmin + rng.randint(1, 4), iterations=rng.randint(4, 24),
                depth=rng.randint(4, 10), compiled=False)


# ---- circuits ---------------------------------------------------------------
# A gate is (target bit, control mask, control value, 2x2 matrix); bit 0 is the
# least significant index bit.

H = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
X = np.array([[0, 1], [1, 0]])
Z = np.diag([1, -1])


def u3(theta, phi, lam):
    c, s = math.cos(theta / 2), math.sin(theta / 2)
    return np.array([[c, -np.exp(1j * lam) * s], [np.exp(1j * phi) * s, np.exp(1j * (phi + lam)) * c]])


def random_gates(n, depth, seed):
    """Layers of a random rotation on every qubit and a brickwork of controlled Z."""
    r = np.random.default_rng(seed)
    for layer in range(depth):
        for b in range(n):
            yield b, 0, 0, u3(*r.uniform(0, 2 * math.pi, 3))
        for b in range(layer % 2, n - 1, 2):
            yield b, 2 << b, 2 << b, Z


def qft_gates(n):
    for b in range(n - 1, -1, -1):
        yield b, 0, 0, H
        for k in range(b - 1, -1, -1):
            yield b, 1 << k, 1 << k, np.diag([1, np.exp(1j * math.pi / (1 << (b - k)))])


def marked(n):
    return int(np.random.default_rng(n).integers(0, 1 << n))


def grover_gates(n, value):
    """One iteration: the oracle's phase flip of `value`, then the inversion about the mean."""
    rest = (1 << n) - 2
    zeros = [b for b in range(n) if not value >> b & 1]
    for b in zeros:
        yield b, 0, 0, X
    yield 0, rest, rest, Z
    for b in zeros:
        yield b, 0, 0, X
    for m in (H, X):
        for b in range(n):
            yield b, 0, 0, m
    yield 0, rest, rest, Z
    for m in (X, H):
        for b in range(n):
            yield b, 0, 0, m


def circuit(case):
    """The case's gate array, as the library takes it, and how often it is applied."""
    n, kind = case["qubits"], case["circuit"]
    if kind == "adder":
        d = hq.DGM()
        d.qubits = n
        d.setFunction(hq.DraperAdder((n - 1) // 2, d))
        return d.ops(), 1
    if kind == "hadamard":
        gates, times = [(b, 0, 0, H) for b in range(n)], case["depth"]
    elif kind == "grover":
        gates, times = grover_gates(n, marked(n)), case["depth"]
    elif kind == "qft":
        gates, times = qft_gates(n), 1
    else:
        gates, times = random_gates(n, case["depth"], n), 1
    return hq.make_ops(*zip(*gates)), times


def tuning(case):
    if case["tuning"] == "default":
        return hq.default_tuning()
    if case["tuning"] == "tile":        # the serving engine's tile: gates fused and row-scaled, interpreted
        return hq.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=4 if case["dtype"] == "c64" else 3,
                                 kernel=N.HGM_KERNEL_REG, planner=N.HGM_PLAN_GREEDY | N.HGM_PLAN_FUSE | N.HGM_PLAN_PIVOT)
    t = N.Tuning()
    N.check(N.lib.hgm_auto_tuning(case["qubits"], CODE[case["dtype"]], C.byref(t)))
    if case["circuit"] == "random":     # the benchmark's planner for layered circuits
        t.planner |= N.HGM_PLAN_LOOKAHEAD
    return t


# ---- inputs -----------------------------------------------------------------

def amplitudes(n, dtype, seed):
    """A normalised state of random amplitudes, on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    a = torch.empty(1 << n, dtype=TORCH[dtype], device="cuda")
    torch.view_as_real(a).normal_(0.0, math.sqrt(0.5) * 2.0 ** (-n / 2), generator=g)
    return a


class Borrowed(hq.State):
    """A state in the caller's device memory (hgm_state_wrap)."""

    def __init__(self, tensor, n, dtype):
        self.dtype, self.qubits, self.tensor = np.dtype(NP[dtype]), n, tensor
        h = C.c_void_p()
        N.check(N.lib.hgm_state_wrap(tensor.data_ptr(), n, CODE[dtype], C.byref(h)))
        self._h = h


def batch_sizes(case):
    span = case["qmax"] - case["qmin"] + 1
    return [case["qmin"] + i % span for i in range(case["states"])]


def requests(case, seed):
    """The requests of a burst: (kind, qubits, parameters). Kinds, sizes and lengths are the case's, the rest the seed's."""
    r, fixed = np.random.default_rng(seed), np.random.default_rng(case["requests"])
    kinds = ("grover",) if case["compiled"] else S.KINDS
    for i in range(case["requests"]):
        n = case["qmin"] + i // len(kinds) % (case["qmax"] - case["qmin"] + 1)
        kind, w = kinds[i % len(kinds)], (n - 1) // 2
        yield kind, n, dict(value=int(r.integers(0, 1 << n)), times=int(fixed.integers(1, case["iterations"] + 1)), seed=int(r.integers(1 << 31)),
                            a=int(r.integers(0, 1 << w)), b=int(r.integers(0, 1 << w)), keep=i % 3 == 2 and not case["compiled"])


def request_gates(case, kind, n, p):
    if kind == "random":
        return list(random_gates(n, case["depth"], p["seed"]))
    return [(b, 0, 0, H) for b in range(n)] + (list(grover_gates(n, p["value"])) * p["times"] if kind == "grover" else [])


def prepare(case, seed):
    kind, dtype = case["kind"], case.get("dtype", "c64")
    st = {"kind": kind}
    if kind == "plan":
        ops, times = circuit(case)
        st["plan"] = hq.Plan(case["qubits"], ops, tuning(case), times, NP[dtype])
    elif kind in ("apply", "execute"):
        st["ops"], st["times"] = circuit(case)
        st["tuning"] = tuning(case)
    if kind in ("plan", "apply", "readout"):
        st["state"] = Borrowed(amplitudes(case["qubits"], dtype, seed), case["qubits"], dtype)
        st["qubit"] = case.get("qubit")
    elif kind == "execute":             # pageable memory, as the reference's state is
        st["host"] = amplitudes(case["qubits"], dtype, seed).cpu().numpy()
        st["qubits"], st["code"] = case["qubits"], CODE[dtype]
    elif kind == "batch":
        sizes = batch_sizes(case)
        st["buffer"] = torch.cat([amplitudes(n, dtype, seed * 1000 + i) for i, n in enumerate(sizes)])
        plans = {n: hq.Plan(n, *batch_circuit(case, n), NP[dtype]) for n in set(sizes)}
        ends = np.cumsum([1 << n for n in sizes])
        st["batch"] = hq.Batch([Borrowed(st["buffer"][e - (1 << n):e], n, dtype) for e, n in zip(ends, sizes)], [plans[n] for n in sizes])
    elif kind == "serve":
        st["server"] = S.Server(np.complex64, hbm_budget_gib=4)
        st["jobs"] = []
        for what, n, p in requests(case, seed):
            basis = 0
            if what == "adder":
                w = (n - 1) // 2
                d = hq.DGM()
                d.setFunction(hq.DraperAdder(w, d))
                ops, basis = S.ops_np(d.ops()), p["a"] << (w + 1) | p["b"]
            else:
                ops = S.ops_np(hq.make_ops(*zip(*request_gates(case, what, n, p))))
            st["jobs"].append((what, n, ops, basis, np.zeros(1 << n, np.complex64) if p["keep"] else None))
        if case["compiled"]:
            for n in range(case["qmin"], case["qmax"] + 1):
                for times in (1, 2, 3, 4):
                    shape = request_gates(case, "grover", n, dict(value=(1 << n) - 1, times=times))
                    st["server"].precompile(n, S.ops_np(hq.make_ops(*zip(*shape))))
    torch.cuda.synchronize()            # the library runs on a stream of its own
    return st


def batch_circuit(case, n):
    """Gate array, tuning and iterations of the batch's states of n qubits: gates fused, compiled kernels."""
    t = hq.default_tuning(block_size=256, repeat_count=8, gpu_region_bits=12, gpu_coalesced_bits=4 if case["dtype"] == "c64" else 3,
                          kernel=N.HGM_KERNEL_JIT, planner=N.HGM_PLAN_GREEDY | N.HGM_PLAN_FUSE, ops_block=1 << 30)
    return hq.make_ops(*zip(*grover_gates(n, marked(n)))), t, case["depth"]


def run(st):
    kind = st["kind"]
    if kind == "plan":
        st["plan"].run(st["state"])
        return st["state"].tensor
    if kind == "apply":
        st["state"].apply(st["ops"], st["tuning"], st["times"])
        return st["state"].tensor
    if kind == "execute":
        N.check(N.lib.hgm_execute(st["host"].ctypes.data, st["qubits"], st["code"], st["ops"], len(st["ops"]), C.byref(st["tuning"]), st["times"],
                                  None))
        return st["host"]
    if kind == "readout":
        s, q = st["state"], st["qubit"]
        zero, one = s.prob_halves(q)
        s.collapse_reset(q, int(one > zero), max(zero, one))
        index, top = s.argmax()
        return {"probabilities": np.array([zero, one]), "index": index, "top": np.array([top]), "norm": np.array([s.norm2()]), "state": s.tensor}
    if kind == "batch":
        st["batch"].run()
        return st["buffer"]
    server, slot, got = st["server"], {}, {}
    for k, (what, n, ops, basis, out) in enumerate(st["jobs"]):
        slot[server.submit(n, ops, basis, state_out=out)] = k
    while len(got) < len(slot):
        for r in server.poll(timeout_ms=1000):
            got[slot[r["id"]]] = r
    rows = [got[k] for k in range(len(slot))]
    for r in rows:
        if r["status"]:
            raise RuntimeError(f"request failed: {r}")
    # a Hadamard layer from |0> has no largest amplitude
    index = [-1 if j[0] == "hadamard" else r["argmax"] for j, r in zip(st["jobs"], rows)]
    out = {"index": np.array(index), "top": np.array([r["p_max"] for r in rows], np.float32), "norm": np.array([r["norm2"] for r in rows], np.float32)}
    kept = [j[4] for j in st["jobs"] if j[4] is not None]
    if kept:
        out["states"] = np.concatenate(kept)
    return out


# ---- what a pass cannot do without, and its values in 64 bits -----------------

def rotations(case, n):
    """Gates that mix amplitudes, after everything that a gate list lets be merged: one per qubit and layer."""
    kind = case["circuit"]
    return n * {"random": case["depth"], "grover": 2 * case["depth"], "adder": 1, "hadamard": 1, "qft": 1}[kind]


def work(case):
    """The state is read once and written once; a merged real rotation costs 4 multiply-adds per amplitude pair."""
    kind, size = case["kind"], 16 if case.get("dtype") == "c128" else 8
    if kind == "readout":
        return {"bytes": 2 * size << case["qubits"], "flops": 6 << case["qubits"]}
    if kind == "batch":
        sizes = batch_sizes(case)
        return {"bytes": sum(2 * size << n for n in sizes), "flops": sum((4 << n) * 2 * n * case["depth"] for n in sizes)}
    if kind == "serve":
        n = (case["qmin"] + case["qmax"]) / 2
        layers = 1 + case["iterations"] if case["compiled"] else (3 + case["iterations"] + case["depth"]) / 4
        return {"bytes": case["requests"] * 2 * size * 2.0 ** n, "flops": case["requests"] * 4 * 2.0 ** n * n * layers}
    return {"bytes": 2 * size << case["qubits"], "flops": (4 << case["qubits"]) * rotations(case, case["qubits"])}


def apply_gate(a, n, target, mask, value, m):
    """One gate on a complex128 state, in place; a gate's untouched amplitudes are not read."""
    bits = sorted([target] + [b for b in range(n) if mask >> b & 1], reverse=True)
    shape, at, last = [], [], n
    for b in bits:
        shape += [1 << (last - 1 - b), 2]
        at += [slice(None), None if b == target else (value >> b & 1)]
        last = b
    v = a.view(shape + [1 << last])
    pick = [v[tuple(t if i is None else i for i in at)] for t in (0, 1)]
    m = np.asarray(m, np.complex128)
    if m[0, 1] == 0 and m[1, 0] == 0:
        for t in (0, 1):
            if m[t, t] != 1:
                pick[t].mul_(complex(m[t, t]))
        return
    zero = pick[0] * complex(m[0, 0])
    zero.add_(pick[1], alpha=complex(m[0, 1]))
    pick[1].mul_(complex(m[1, 1])).add_(pick[0], alpha=complex(m[1, 0]))
    pick[0].copy_(zero)


def evolve(a, n, kind, depth, value=None, seed=None):
    if kind == "grover":                # X..Z..X, H X..Z..X H = I - 2|s><s|
        for _ in range(depth):
            a[value].neg_()
            a.sub_(2 * a.mean())
        return a
    if kind == "adder":                 # |a, b> -> |a, a + b mod 2^(w+1)>
        w = (n - 1) // 2
        row = torch.arange(1 << w, device=a.device)[:, None]
        col = torch.arange(2 << w, device=a.device)[None, :]
        v, out = a.view(1 << w, 2 << w), torch.empty_like(a).view(1 << w, 2 << w)
        for k in range(0, 1 << w, 1024):
            out[k:k + 1024] = v[k:k + 1024].gather(1, (col - row[k:k + 1024]) % (2 << w))
        return out.view(-1)
    gates = {"random": lambda: random_gates(n, depth, n if seed is None else seed), "qft": lambda: qft_gates(n),
             "hadamard": lambda: [(b, 0, 0, H) for b in range(n)] * depth}[kind]()
    for g in gates:
        apply_gate(a, n, *g)
    return a


def exact(case, seed):
    kind, dtype = case["kind"], case.get("dtype", "c64")
    if kind in ("plan", "apply", "execute"):
        a = evolve(amplitudes(case["qubits"], dtype, seed).to(torch.complex128), case["qubits"], case["circuit"], case["depth"], marked(case["qubits"]))
        return a.cpu().numpy() if kind == "execute" else a
    if kind == "readout":
        n, q = case["qubits"], case["qubit"]
        v = amplitudes(n, dtype, seed).to(torch.complex128).view(1 << q, 2, -1)
        zero, one = (float(torch.view_as_real(v[:, t]).square().sum()) for t in (0, 1))
        v[:, 0] = v[:, int(one > zero)] / math.sqrt(max(zero, one))
        v[:, 1] = 0
        p = torch.view_as_real(v).square().sum(-1).view(-1)
        return {"probabilities": np.array([zero, one]), "index": None, "top": np.array([float(p.max())]), "norm": np.array([float(p.sum())]),
                "state": v.reshape(-1)}
    if kind == "batch":
        return torch.cat([evolve(amplitudes(n, dtype, seed * 1000 + i).to(torch.complex128), n, "grover", case["depth"], marked(n))
                          for i, n in enumerate(batch_sizes(case))])
    top, norm, kept = [], [], []
    for what, n, p in requests(case, seed):
        a = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
        if what == "adder":
            w = (n - 1) // 2
            a[p["a"] << (w + 1) | (p["a"] + p["b"])] = 1
        else:
            a[0] = 1
            if what == "random":
                evolve(a, n, "random", case["depth"], seed=p["seed"])
            else:
                a.fill_(2.0 ** (-n / 2))
                evolve(a, n, "grover", p["times"] if what == "grover" else 0, p["value"])
        q = torch.view_as_real(a).square().sum(-1)
        top.append(float(q.max()))
        norm.append(float(q.sum()))
        if p["keep"]:
            kept.append(a.cpu().numpy())
    out = {"index": None, "top": np.array(top), "norm": np.array(norm)}
    if kept:
        out["states"] = np.concatenate(kept)
    return out
