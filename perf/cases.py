"""Timed cases of the engine: whole programs through its public entry points (graph runs, the StateType
backends, the batching form), over the sizes they are used at.

A case is a dict with a "kind" and its sizes:

  qft      the graph frontend: run(StochasticMeasure(QFFT(q)), feed={q: psi}) on n qubits. Small states,
           where launches and the host's work per gate count; the program reads the state and its
           probabilities.
  circuit  a layered random circuit (Haar gates on every qubit, then CNOT or CZ bricks) applied descriptor
           by descriptor from |0...0> on one of the four forms: plain128 and plain64 (gate by gate), fused64
           (split-BF16 MFMA blocks) and fused128 (FP64 blocks). Up to 20 qubits the program reads the whole
           state, above that the joint distribution of its first 20 qubits. The complex64 forms' figures
           are kept in single precision, the precision of their states.
  grover   iterations of Grover's search (a table oracle, H and X layers, a many-controlled Z) from the
           uniform state; the program reads the most likely outcome and the distribution of up to 16 of
           the search qubits.
  order    order finding: |x>|0> -> |x>|a^x mod N> from a fed register, measurement of the second
           register, the quantum Fourier transform of the first, and its distribution.
  dense    wide unitaries (4 to 8 qubits, one under a control) on a large complex128 state.
  batch    many small circuits of uneven sizes run together, every state read.
"""
import math

import numpy
import torch

from qip_amd import CMat, FuncTable, GpuBackend, QFFT, Qubit, StochasticMeasure, run as run_graph
from qip_amd.batch import GpuBatch, PackedCircuits
from qip_amd.fused import Fused128Backend, FusedBackend
from qip_amd.workloads import (apply_ops, grover_initial, grover_iteration_ops, grover_iterations,
                               layered_circuit_gates, layered_random_circuit)

FORMS = {"plain128": (GpuBackend, numpy.complex128), "plain64": (GpuBackend, numpy.complex64),
         "fused64": (FusedBackend, numpy.complex64), "fused128": (Fused128Backend, numpy.complex128)}
READ_STATE = 20      # qubits up to which a circuit's whole state is read
READ_QUBITS = 20     # qubits of the joint distribution read above that
SEARCH_READ = 16     # search qubits whose distribution a search reads
MODULI = ((3, 2), (5, 2), (15, 7), (21, 2), (55, 3), (119, 5), (221, 7))   # (N, a), a coprime to N


def listed():
    return [
        # the smallest whole call: a few hundred kilobytes, bound by launches and host work
        {"name": "qft_graph_10", "kind": "qft", "n": 10},
        # the 16-qubit Fourier transform of the benchmark
        {"name": "qft_graph_16", "kind": "qft", "n": 16},
        # an ordinary circuit on the drop-in backend, state in cache, whole state read
        {"name": "circuit_plain128_20", "kind": "circuit", "form": "plain128", "n": 20, "depth": 16},
        # the 28-qubit depth-20 circuit of the benchmark on the drop-in backend
        {"name": "circuit_plain128_28", "kind": "circuit", "form": "plain128", "n": 28, "depth": 20},
        # an unfused complex64 circuit of odd size
        {"name": "circuit_plain64_27", "kind": "circuit", "form": "plain64", "n": 27, "depth": 17},
        # the 30-qubit depth-40 circuit of the benchmark in the precision form
        {"name": "circuit_fused64_30", "kind": "circuit", "form": "fused64", "n": 30, "depth": 40},
        # the same blocks in FP64
        {"name": "circuit_fused128_27", "kind": "circuit", "form": "fused128", "n": 27, "depth": 20},
        # the 24-qubit search of the benchmark, drop-in and precision form
        {"name": "grover_plain128_24", "kind": "grover", "form": "plain128", "ns": 23, "iters": 40},
        {"name": "grover_fused64_24", "kind": "grover", "form": "fused64", "ns": 23, "iters": 80},
        # order finding modulo 221 with a 19-qubit first register
        {"name": "order_finding_27", "kind": "order", "n1": 19, "n2": 8, "low": False},
        # wide unitaries on 1 GiB
        {"name": "dense_26", "kind": "dense", "n": 26, "ks": "4,5,6,6,7,8"},
        # small circuits served together
        {"name": "batch_48", "kind": "batch", "count": 48, "n_lo": 10, "n_hi": 20, "d_lo": 8, "d_hi": 32},
    ]


def draw(rng):
    kind = rng.choice(["qft", "circuit", "circuit", "circuit", "grover", "order", "dense", "batch"])
    if kind == "qft":
        return {"kind": kind, "n": rng.randint(5, 18)}
    if kind == "circuit":
        form = rng.choice(sorted(FORMS))
        top = {"plain128": 27, "plain64": 28, "fused64": 29, "fused128": 27}[form]
        return {"kind": kind, "form": form, "n": rng.randint(9, top), "depth": rng.randint(5, 20)}
    if kind == "grover":
        ns = rng.randint(9, 23)
        return {"kind": kind, "form": rng.choice(sorted(FORMS)), "ns": ns,
                "iters": rng.randint(4, min(40, grover_iterations(ns)))}
    if kind == "order":
        n2 = rng.randint(2, 8)
        return {"kind": kind, "n1": rng.randint(8, 26 - n2), "n2": n2, "low": rng.random() < 0.5}
    if kind == "dense":
        ks = ",".join(str(rng.randint(4, 8)) for _ in range(rng.randint(2, 6)))
        return {"kind": kind, "n": rng.randint(13, 26), "ks": ks}
    lo = rng.randint(8, 13)
    return {"kind": kind, "count": rng.randint(5, 48), "n_lo": lo, "n_hi": rng.randint(lo + 1, 20),
            "d_lo": rng.randint(4, 12), "d_hi": rng.randint(13, 32)}


def _unit(rng, count):
    v = rng.standard_normal(count) + 1j * rng.standard_normal(count)
    return v / numpy.linalg.norm(v)


def _unitary(rng, dim):
    z = rng.standard_normal((dim, dim)) + 1j * rng.standard_normal((dim, dim))
    q, r = numpy.linalg.qr(z)
    d = numpy.diagonal(r)
    return q * (d / numpy.abs(d))


def _marked(case, rng):
    return int(rng.integers(0, 2 ** case["ns"]))


def _modulus(case):
    return [m for m in MODULI if m[0] <= 2 ** case["n2"] - 1][-1]


def _order_setup(case, seed):
    """(first register, second register, its function's values, the fed vector, the outcome measured)."""
    rng = numpy.random.default_rng(seed)
    n1, n2 = case["n1"], case["n2"]
    N, a = _modulus(case)
    period = [1]
    while period[-1] * a % N != 1:
        period.append(period[-1] * a % N)
    values = numpy.array(period, dtype=numpy.int64)[numpy.arange(2 ** n1) % len(period)]
    psi = _unit(rng, 2 ** n1)
    outcome = int(values[int(rng.integers(0, 2 ** n1))])
    reg1, reg2 = (list(range(n2, n1 + n2)), list(range(n2))) if case["low"] else \
        (list(range(n1)), list(range(n1, n1 + n2)))
    return reg1, reg2, values, psi, outcome


def _qft_ops(reg):
    h = numpy.array([[1.0, 1.0], [1.0, -1.0]]) / numpy.sqrt(2.0)
    swap = numpy.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], dtype=numpy.complex128)
    ops = []
    for t in range(len(reg)):
        ops.append({reg[t]: h})
        for i in range(t + 1, len(reg)):
            phase = numpy.exp(2j * numpy.pi / 2.0 ** (1 + i - t))
            ops.append({(reg[i], reg[t]): CMat(numpy.array([[1, 0], [0, phase]]))})
    for i in range(len(reg) // 2):
        ops.append({(reg[i], reg[-1 - i]): swap})
    return ops


def _bit_order(value, k):
    """The place of a k-qubit register's value (first qubit = highest bit) in measure_probabilities' result,
    which has the register's j-th qubit on bit j."""
    return int(format(value, "0{}b".format(k))[::-1], 2)


def _dense_ops(case, seed):
    """[(targets, controls, unitary)]: low, high and scattered targets in turn, every third one under a
    control."""
    rng = numpy.random.default_rng(seed)
    n, out = case["n"], []
    for i, k in enumerate(int(x) for x in case["ks"].split(",")):
        if i % 3 == 0:
            t = list(range(n - k, n))
        elif i % 3 == 1:
            t = list(range(k))
        else:
            t = sorted(int(q) for q in rng.choice(n - 1, k, replace=False) + 1)
        c = [0] if i % 3 == 2 else []
        out.append((t, c, _unitary(rng, 2 ** k)))
    return out


def _batch_circuits(case, seed):
    # the sizes follow from the case alone, spread unevenly over their ranges; the gates from the seed
    sizes = numpy.random.default_rng(case["count"])
    ns = [int(v) for v in sizes.integers(case["n_lo"], case["n_hi"] + 1, size=case["count"])]
    ds = [int(v) for v in sizes.integers(case["d_lo"], case["d_hi"] + 1, size=case["count"])]
    seeds = [int(v) for v in numpy.random.default_rng(seed).integers(0, 2 ** 31 - 1, size=case["count"])]
    ns[0], ns[-1] = case["n_hi"], case["n_lo"]      # both ends of the range are there
    return ns, [layered_circuit_gates(n, d, s) for n, d, s in zip(ns, ds, seeds)]


def prepare(case, seed):
    rng = numpy.random.default_rng(seed)
    kind = case["kind"]
    if kind == "qft":
        q = Qubit(n=case["n"])
        return {"kind": kind, "q": q, "out": StochasticMeasure(QFFT(q)), "psi": _unit(rng, 2 ** case["n"])}
    if kind == "circuit":
        cls, dtype = FORMS[case["form"]]
        be = cls.make_state(case["n"], [], [], statetype=dtype)
        return {"kind": kind, "be": be, "n": case["n"], "dtype": dtype,
                "ops": layered_random_circuit(case["n"], case["depth"], seed)}
    if kind == "grover":
        cls, dtype = FORMS[case["form"]]
        ns = case["ns"]
        groups, feeds = grover_initial(ns)
        be = cls.make_state(ns + 1, groups, feeds, statetype=dtype)
        return {"kind": kind, "be": be, "ns": ns, "dtype": dtype, "groups": groups, "feeds": feeds,
                "ops": grover_iteration_ops(ns, _marked(case, rng), "mcz"), "iters": case["iters"]}
    if kind == "order":
        reg1, reg2, values, psi, outcome = _order_setup(case, seed)
        be = GpuBackend.make_state(case["n1"] + case["n2"], [reg1], [psi])
        return {"kind": kind, "be": be, "reg1": reg1, "reg2": reg2, "f": FuncTable(values), "psi": psi,
                "outcome": outcome, "ops": _qft_ops(reg1)}
    if kind == "dense":
        n = case["n"]
        feeds = [_unit(rng, 2 ** (n // 2)), _unit(rng, 2 ** (n - n // 2))]
        groups = [list(range(n // 2)), list(range(n // 2, n))]
        ops = []
        for t, c, u in _dense_ops(case, seed):
            for _ in c:
                u = CMat(u)
            ops.append({tuple(c + t): u})
        return {"kind": kind, "be": GpuBackend.make_state(n, groups, feeds), "n": n, "groups": groups,
                "feeds": feeds, "ops": ops}
    ns, circuits = _batch_circuits(case, seed)
    b = GpuBatch(ns)
    b.load(PackedCircuits.from_gates(ns, circuits))
    return {"kind": "batch", "b": b}


def _stored(x, dtype):
    """Figures of a complex64 state kept in single precision, of a complex128 one in double."""
    x = numpy.asarray(x)
    return x.astype(numpy.float32) if dtype == numpy.complex64 and x.dtype == numpy.float64 else x


def run(s):
    kind = s["kind"]
    if kind == "qft":
        state, notes = run_graph(s["out"], feed={s["q"]: s["psi"]})
        return {"state": state, "probs": notes[s["out"]]}
    be = s.get("be")
    if kind == "circuit":
        be.reinit()
        for d in s["ops"]:
            be.kronselect_dot(d)
        if s["n"] <= READ_STATE:
            return {"state": be.get_state()}
        return {"probs": _stored(be.measure_probabilities(list(range(READ_QUBITS))), s["dtype"])}
    if kind == "grover":
        be.reinit(s["groups"], s["feeds"])
        for _ in range(s["iters"]):
            apply_ops(be, s["ops"])
        best, p = be.measure_probabilities(list(range(s["ns"])), top_k=1)
        probs = be.measure_probabilities(list(range(min(s["ns"], SEARCH_READ))))
        return {"best": best[0], "p": _stored(p, s["dtype"]), "probs": _stored(probs, s["dtype"])}
    if kind == "order":
        be.reinit([s["reg1"]], [s["psi"]])
        be.func_apply(s["reg1"], s["reg2"], s["f"])
        second = be.measure_probabilities(s["reg2"])
        m, p = be.measure(s["reg2"], measured=s["outcome"])
        for d in s["ops"]:
            be.kronselect_dot(d)
        return {"second": second, "m": m, "p": p, "first": be.measure_probabilities(s["reg1"])}
    if kind == "dense":
        be.reinit(s["groups"], s["feeds"])
        for d in s["ops"]:
            be.kronselect_dot(d)
        if s["n"] <= READ_STATE:
            return {"state": be.get_state()}
        return {"probs": be.measure_probabilities(list(range(READ_QUBITS))), "norm": be.total_prob()}
    b = s["b"]
    b.reset()
    b.run()
    return {"states": [b.get_state(i) for i in range(b.count)]}


def _gates(n, depth):
    """(Haar gates, CNOTs, CZs) of a layered circuit."""
    return n * depth, (depth + 1) // 2 * (n // 2), depth // 2 * ((n - 1) // 2)


def work(case):
    """The state written once and read once, the inputs and outputs once; 14 flops an amplitude for a
    single-qubit gate, 6 for half of them for a phase, 8 D for a dense operator on D = 2^k rows."""
    kind = case["kind"]
    if kind == "qft":
        n = case["n"]
        return {"bytes": 2 * 16 * 2 ** n + 8 * 2 ** n, "flops": 2 ** n * (14 * n + 6 * n * (n - 1) / 8)}
    if kind == "circuit":
        n = case["n"]
        amp = 16 if case["form"].endswith("128") else 8
        one, _, _ = _gates(n, case["depth"])
        out = amp * 2 ** n if n <= READ_STATE else (amp // 2) * 2 ** READ_QUBITS
        return {"bytes": 2 * amp * 2 ** n + out, "flops": 14.0 * one * 2 ** n}
    if kind == "grover":
        ns, amp = case["ns"], 16 if case["form"].endswith("128") else 8
        return {"bytes": case["iters"] * 4 * 2 ** ns + 2 * amp * 2 ** (ns + 1),
                "flops": 2 ** (ns + 1) * case["iters"] * 2.0 * 4 * ns}
    if kind == "order":
        n1, n = case["n1"], case["n1"] + case["n2"]
        return {"bytes": 16 * 2 ** n1 + 2 * 16 * 2 ** n + 8 * 2 ** n1 + 4 * 2 ** n1,
                "flops": 2 ** n * (14.0 * n1 + 6 * n1 * (n1 - 1) / 8)}
    if kind == "dense":
        ks = [int(x) for x in case["ks"].split(",")]
        fl = sum((0.5 if i % 3 == 2 else 1.0) * 8 * 2 ** k for i, k in enumerate(ks))
        return {"bytes": 2 * 16 * 2 ** case["n"], "flops": fl * 2 ** case["n"]}
    lo, hi = case["n_lo"], case["n_hi"]
    amps = case["count"] * (2 ** (hi + 1) - 2 ** lo) / (hi - lo + 1)
    return {"bytes": 2 * 8 * amps, "flops": 14.0 * amps * (lo + hi) / 2 * (case["d_lo"] + case["d_hi"]) / 2}


# ---- 64-bit values in plain torch ------------------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _dev(x):
    return torch.as_tensor(numpy.ascontiguousarray(x), dtype=torch.complex128).to(_DEV)


def _axes(n, qubits):
    """A shape for 2^n amplitudes with an axis of its own for each of the ascending qubits, and those
    axes."""
    shape, axes, at = [], [], 0
    for q in qubits:
        if q > at:
            shape.append(2 ** (q - at))
        axes.append(len(shape))
        shape.append(2)
        at = q + 1
    if at < n:
        shape.append(2 ** (n - at))
    return shape, axes


def _apply(v, n, qubits, u):
    """u on the ascending qubits (first = highest bit of its index) of the 2^n amplitudes v."""
    shape, axes = _axes(n, qubits)
    rest = [a for a in range(len(shape)) if a not in axes]
    order = axes + rest
    x = v.view(shape).permute(order).reshape(2 ** len(qubits), -1)
    x = u @ x
    back = [order.index(a) for a in range(len(shape))]
    return x.view([shape[a] for a in order]).permute(back).reshape(-1).contiguous()


def _kron(mats):
    out = numpy.ones((1, 1), dtype=numpy.complex128)
    for m in mats:
        out = numpy.kron(out, m)
    return out


def _layered(n, gates):
    """The layered circuit on |0...0>: each run of single-qubit gates as products on up to six leading
    qubits at a time, the register turned by their width after each."""
    v = torch.zeros(2 ** n, dtype=torch.complex128, device=_DEV)
    v[0] = 1
    i = 0
    while i < len(gates):
        ones = []
        while i < len(gates) and len(gates[i][0]) == 1:
            ones.append(gates[i][1])
            i += 1
        for lo in range(0, n, 6):
            w = min(6, n - lo)
            x = _dev(_kron(ones[lo:lo + w])) @ v.view(2 ** w, -1)
            v = x.t().contiguous().view(-1)
            del x
        while i < len(gates) and len(gates[i][0]) == 2:
            (c, t), g = gates[i]
            i += 1
            shape, axes = _axes(n, [c, t])
            x = v.view(shape)
            one = [slice(None)] * len(shape)
            one[axes[0]] = 1
            if g[3, 3] == -1:
                one[axes[1]] = 1
                x[tuple(one)] *= -1
            else:
                lo_, hi_ = list(one), list(one)
                lo_[axes[1]], hi_[axes[1]] = 0, 1
                keep = x[tuple(lo_)].clone()
                x[tuple(lo_)] = x[tuple(hi_)]
                x[tuple(hi_)] = keep
    return v


def _probs(v, n, k):
    """The distribution of the first k qubits, qubit j on bit j, as measure_probabilities gives it."""
    p = torch.empty(2 ** k, dtype=torch.float64, device=v.device)
    rows, step = v.view(2 ** k, -1), max(1, 2 ** 26 // 2 ** (n - k))
    for lo in range(0, 2 ** k, step):
        x = torch.view_as_real(rows[lo:lo + step])
        p[lo:lo + step] = x.square().sum(dim=(1, 2))
    return _reversed(p.cpu().numpy(), k)


def _reversed(p, k):
    return numpy.ascontiguousarray(p.reshape([2] * k).transpose(list(range(k))[::-1])).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    rng = numpy.random.default_rng(seed)
    if kind == "qft":
        n = case["n"]
        state = numpy.fft.ifft(_unit(rng, 2 ** n), norm="ortho")
        return {"state": state, "probs": _reversed(numpy.abs(state) ** 2, n)}
    if kind == "circuit":
        n = case["n"]
        v = _layered(n, layered_circuit_gates(n, case["depth"], seed))
        return {"state": v.cpu().numpy()} if n <= READ_STATE else {"probs": _probs(v, n, READ_QUBITS)}
    if kind == "grover":
        ns, t, x = case["ns"], case["iters"], _marked(case, rng)
        theta = math.asin(2.0 ** (-ns / 2))
        p = numpy.full(2 ** ns, math.cos((2 * t + 1) * theta) ** 2 / (2 ** ns - 1))
        p[x] = math.sin((2 * t + 1) * theta) ** 2
        k = min(ns, SEARCH_READ)
        return {"best": None, "p": float(p.max()),
                "probs": _reversed(p.reshape(2 ** k, -1).sum(axis=1), k)}
    if kind == "order":
        _, _, values, psi, outcome = _order_setup(case, seed)
        w = numpy.abs(psi) ** 2
        second = numpy.zeros(2 ** case["n2"])
        by = numpy.bincount(values, weights=w, minlength=2 ** case["n2"])
        for y in range(2 ** case["n2"]):
            second[_bit_order(y, case["n2"])] = by[y]
        p = by[outcome]
        left = numpy.where(values == outcome, psi, 0) / math.sqrt(p)
        first = numpy.abs(numpy.fft.ifft(left, norm="ortho")) ** 2
        return {"second": second, "m": None, "p": float(p), "first": _reversed(first, case["n1"])}
    if kind == "dense":
        n = case["n"]
        v = torch.outer(_dev(_unit(rng, 2 ** (n // 2))), _dev(_unit(rng, 2 ** (n - n // 2)))).reshape(-1)
        for t, c, u in _dense_ops(case, seed):
            if c:       # qubit 0: the upper half of the state
                v[2 ** (n - 1):] = _apply(v[2 ** (n - 1):].clone(), n - 1, [q - 1 for q in t], _dev(u))
            else:
                v = _apply(v, n, t, _dev(u))
        if n <= READ_STATE:
            return {"state": v.cpu().numpy()}
        return {"probs": _probs(v, n, READ_QUBITS), "norm": 1.0}
    ns, circuits = _batch_circuits(case, seed)
    return {"states": [_layered(n, g).cpu().numpy() for n, g in zip(ns, circuits)]}
