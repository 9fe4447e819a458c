"""Workloads of the state-vector engine, for timing it as a program uses it.

A case names a kind of work and its sizes.  ``prepare`` builds what a program
holds before the call (a circuit handle, a gate list, a batch), ``run`` takes
one pass through the package's public entry points, from |0...0> to what the
program reads back: amplitudes where they are few, shots, measured bits or the
most likely state where they are not.  Shots and measurements draw from
rand(), seeded at the start of each pass, as a reproducible run does.

Kinds:
  plain    layered circuit (H, then layers of RZ RY RZ and two CNOT ladders),
           gate by gate in complex128, or complex64 with "fp32"
  qft      a Fourier state (H and one phase per qubit), the QFT with final
           swaps, then shots: the read-out of phase estimation
  grover   search of one marked index, then the most likely state
  measure  a shallow layered circuit, then qc_measure_all
  fused    layered circuit in the fused complex64 form, one HBM pass per block
           or, with "tiles", as tile programs
  batch    many small circuits (every second one fused) in one launch
"""
import math

import numpy as np
import torch

import qcs_amd
from qcs_amd import circuits as C


def listed():
    return [
        # the smallest circuits a program steps through: launches and latency
        {"name": "plain_10q", "kind": "plain", "n": 10, "depth": 8, "fp32": False, "out": "read"},
        # an ordinary circuit whose state the program reads back
        {"name": "plain_17q", "kind": "plain", "n": 17, "depth": 12, "fp32": False, "out": "read"},
        # the 20-qubit, depth-10 circuit and its 1024-shot histogram
        {"name": "plain_20q", "kind": "plain", "n": 20, "depth": 10, "fp32": False, "out": "hist"},
        # the plain form at a size where only shots come back
        {"name": "plain_28q", "kind": "plain", "n": 28, "depth": 6, "fp32": False, "out": "shots"},
        # the plain form in complex64, an odd size
        {"name": "plain32_25q", "kind": "plain", "n": 25, "depth": 9, "fp32": True, "out": "shots"},
        # phase estimation's read-out at the 28-qubit QFT's size
        {"name": "qft_28q", "kind": "qft", "n": 28, "out": "shots"},
        # a whole search: 100 rounds on a small state
        {"name": "grover_14q", "kind": "grover", "n": 14, "rounds": 0, "out": "read"},
        # a truncated search on a large state
        {"name": "grover_27q", "kind": "grover", "n": 27, "rounds": 16, "out": "best"},
        # qc_run: a state collapsed qubit by qubit
        {"name": "measure_26q", "kind": "measure", "n": 26, "depth": 1},
        # the fused form's default (one HBM pass per block), state read back
        {"name": "fused_18q", "kind": "fused", "n": 18, "depth": 10, "tiles": False, "out": "read"},
        # the 30-qubit, depth-20 circuit as tile programs
        {"name": "fused_30q", "kind": "fused", "n": 30, "depth": 20, "tiles": True, "out": "shots"},
        # small circuits of mixed sizes, planned and run together
        {"name": "batch_256", "kind": "batch", "count": 256, "lo": 10, "hi": 18, "dlo": 5, "dhi": 40},
    ]


def _depth(rng, n, most_updates, most):
    """A depth, spread over its logarithm, whose amplitude updates stay below
    ``most_updates``."""
    top = max(1, min(most, int(most_updates / (4.0 * n * 2.0 ** n))))
    return max(1, min(top, int(round(math.exp(rng.uniform(0.0, math.log(top + 0.5)))))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "qft", "grover", "measure", "fused", "fused", "batch"])
    if kind == "plain":
        n = rng.randint(8, 28)
        out = rng.choice(["read", "hist"]) if n <= 18 else "hist" if n <= 21 else "shots"
        return {"kind": "plain", "n": n, "depth": _depth(rng, n, 1.4e11, 24),
                "fp32": rng.random() < 0.3, "out": out}
    if kind == "qft":
        n = rng.randint(8, 28)
        return {"kind": "qft", "n": n, "out": "read" if n <= 18 and rng.random() < 0.5 else "shots"}
    if kind == "grover":
        n = rng.randint(8, 27)
        whole = n <= 20 and rng.random() < 0.6
        return {"kind": "grover", "n": n, "rounds": 0 if whole else rng.randint(2, 24),
                "out": "read" if n <= 18 else "best"}
    if kind == "measure":
        return {"kind": "measure", "n": rng.randint(8, 26), "depth": rng.randint(1, 2)}
    if kind == "fused":
        tiles = rng.random() < 0.5
        n = rng.randint(16, 30) if tiles else rng.randint(8, 27)
        return {"kind": "fused", "n": n, "depth": _depth(rng, n, 2.5e12 if tiles else 2.5e11, 24),
                "tiles": tiles, "out": "read" if n <= 18 else "shots"}
    lo = rng.randint(8, 14)
    dlo = rng.randint(2, 16)
    return {"kind": "batch", "count": rng.randint(24, 256), "lo": lo, "hi": lo + rng.randint(1, 4),
            "dlo": dlo, "dhi": dlo + rng.randint(2, 20)}


_SHOTS = 1024


def _rounds(case):
    return case["rounds"] or int(math.floor(math.pi / 4.0 * math.sqrt(2.0 ** case["n"])))


def _marked(case, seed):
    return int(next(C.splitmix64(seed ^ 0x6D61726B)) % (1 << case["n"]))


def _qft_ops(n, seed):
    """|x> -> exp(-2 pi i phi x) / sqrt(N) for a phase phi from the seed (the
    QFT below takes qubit 0 as the most significant bit), then the QFT."""
    phi = C.uniforms(seed, 1)[0]
    ops = C.Ops()
    for q in range(n):
        ops.add(C.H, q)
    for q in range(n):
        ops.add(C.P, q, -1, -2.0 * math.pi * ((phi * 2.0 ** (n - 1 - q)) % 1.0))
    body = C.qft(n, swaps=True)
    for op, t, c, p in zip(body.op, body.tq, body.cq, body.par):
        ops.add(op, t, c, p)
    return ops


def _ops(case, seed):
    if case["kind"] == "qft":
        return _qft_ops(case["n"], seed)
    return C.layered(case["n"], case["depth"], seed)


def _options(case):
    if case["kind"] == "fused":
        return qcs_amd.FUSED_FP32 | (qcs_amd.FUSE_TILES if case["tiles"] else 0)
    return qcs_amd.PLAIN_FP32 if case.get("fp32") else qcs_amd.PLAIN_FP64


class _State:
    """What a program has in hand: handles, gate list, seed."""

    def __init__(self, case, seed):
        self.case, self.seed, self.libc = case, seed & 0x7FFFFFFF, qcs_amd.libc()
        self.circuits, self.batch = [], None

    def __del__(self):
        if self.batch is not None:
            self.batch.close()
        for c in self.circuits:
            c.close()


def prepare(case, seed):
    s = _State(case, seed)
    if case["kind"] == "batch":
        work = C.batch_workload(case["count"], seed, (case["lo"], case["hi"]),
                                (case["dlo"], case["dhi"]))
        for n, depth, cseed, fused in work:
            c = qcs_amd.Circuit(n, qcs_amd.DEFERRED | (qcs_amd.FUSED_FP32 if fused else 0))
            c.apply(C.layered(n, depth, cseed))
            s.circuits.append(c)
        # every pass plans, as it would for circuits it has not seen
        s.batch = qcs_amd.Batch(qcs_amd.BATCH_REPLAN)
        return s
    s.circuits.append(qcs_amd.Circuit(case["n"], _options(case)))
    if case["kind"] == "grover":
        s.marked, s.rounds = _marked(case, seed), _rounds(case)
    else:
        s.ops = _ops(case, seed)
    return s


def run(s):
    case = s.case
    s.libc.srand(s.seed)
    if case["kind"] == "batch":
        return s.batch.sample(s.circuits, 256)
    c = s.circuits[0]
    c.set_basis_state(0)
    if case["kind"] == "grover":
        c.grover_search_iters(s.marked, s.rounds)
        best = c.find_most_likely_state_l()
        if case["out"] == "read":
            return {"best": best, "amplitudes": c.amplitudes()}
        return {"best": best, "probability": c.get_probability_l(s.marked)}
    c.apply(s.ops)
    if case["kind"] == "measure":
        return np.array(c.measure_all_list())
    if case["out"] == "read":
        a = c.amplitudes()
        # a complex64 state is read as doubles; its own type holds all of it
        return a.astype(np.complex64) if _options(case) != qcs_amd.PLAIN_FP64 else a
    if case["out"] == "hist":
        return c.run_shots_hist(_SHOTS)
    return c.sample_indices(_SHOTS)


def _gate_flops(ops, n):
    """Multiplies and adds the gates need: a real 2x2 or a diagonal costs 6 per
    amplitude it changes, an exchange none."""
    per = {C.H: 6.0, C.RY: 6.0, C.RX: 6.0, C.RZ: 6.0, C.P: 3.0, C.Z: 0.5, C.CPHASE: 1.5}
    return sum(per.get(op, 0.0) for op in ops.op) * 2.0 ** n


def work(case):
    if case["kind"] == "batch":
        b = f = 0.0
        for n, depth, _, fused in C.batch_workload(case["count"], 1, (case["lo"], case["hi"]),
                                                   (case["dlo"], case["dhi"])):
            # the state is read once by the sampling; shots go in and out
            b += 2.0 ** n * (8 if fused else 16) + 256 * 16
            f += (6.0 * n + 18.0 * n * depth) * 2.0 ** n
        return {"bytes": b, "flops": f}
    n = case["n"]
    amp = 2.0 ** n * (8 if case.get("fp32") or case["kind"] == "fused" else 16)
    if case["kind"] == "grover":
        # the state written once and read once, two operations per component
        # and round (the sum, the reflection)
        return {"bytes": 2.0 * amp, "flops": 4.0 * _rounds(case) * 2.0 ** n}
    flops = _gate_flops(_ops(case, 1), n)
    if case["kind"] == "measure":
        return {"bytes": 3.0 * amp, "flops": flops + 6.0 * 2.0 ** n}
    out = 2.0 ** n * 16 if case["out"] == "read" else 2.0 ** n * 4 if case["out"] == "hist" else _SHOTS * 16.0
    return {"bytes": 2.0 * amp + out, "flops": flops}


def _simulate(ops, n):
    """The gates one after another in complex128."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    a = torch.zeros(1 << n, dtype=torch.complex128, device=dev)
    a[0] = 1.0
    r = 1.0 / math.sqrt(2.0)
    for op, t, c, p in zip(ops.op, ops.tq, ops.cq, ops.par):
        if op in (C.CNOT, C.CPHASE, C.SWAP):
            lo, hi = min(t, c), max(t, c)
            v = a.view(1 << (n - 1 - hi), 2, 1 << (hi - lo - 1), 2, 1 << lo)
            if op == C.CPHASE:
                v[:, 1, :, 1, :] *= complex(math.cos(p), math.sin(p))
            elif op == C.SWAP:
                x = v[:, 0, :, 1, :].clone()
                v[:, 0, :, 1, :] = v[:, 1, :, 0, :]
                v[:, 1, :, 0, :] = x
            else:
                one = v[:, 1] if c == hi else v[:, :, :, 1]
                x = (one[:, :, 0, :] if c == hi else one[:, 0]).clone()
                if c == hi:
                    one[:, :, 0, :] = one[:, :, 1, :]
                    one[:, :, 1, :] = x
                else:
                    one[:, 0] = one[:, 1]
                    one[:, 1] = x
            continue
        v = a.view(1 << (n - 1 - t), 2, 1 << t)
        x, y = v[:, 0].clone(), v[:, 1].clone()
        if op == C.H:
            v[:, 0], v[:, 1] = r * x + r * y, r * x - r * y
        elif op == C.RY:
            v[:, 0] = math.cos(p / 2) * x - math.sin(p / 2) * y
            v[:, 1] = math.sin(p / 2) * x + math.cos(p / 2) * y
        elif op == C.RZ:
            v[:, 0] = complex(math.cos(p / 2), -math.sin(p / 2)) * x
            v[:, 1] = complex(math.cos(p / 2), math.sin(p / 2)) * y
        elif op == C.P:
            v[:, 1] = complex(math.cos(p), math.sin(p)) * y
        else:
            raise ValueError(f"gate {op} is not part of these circuits")
    return a.cpu().numpy()


def exact(case, seed):
    if case["kind"] == "grover":
        n, m, k = case["n"], _marked(case, seed), _rounds(case)
        N = 2.0 ** n
        theta = math.asin(1.0 / math.sqrt(N))
        hit = math.sin((2 * k + 1) * theta)
        if case["out"] != "read":
            return {"best": None, "probability": hit * hit}
        a = np.full(1 << n, math.cos((2 * k + 1) * theta) / math.sqrt(N - 1.0), np.complex128)
        a[m] = hit
        return {"best": None, "amplitudes": a}
    if case.get("out") != "read":
        return None  # shots, histograms and measured bits are whole numbers
    return _simulate(_ops(case, seed), case["n"])
