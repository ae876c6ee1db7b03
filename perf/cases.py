"""Timed workloads of the framework, through its Python entry points.

Each case is one pass of something a program built on this framework does:
run a circuit on a resident state and read it out, apply single gates, permute
axes, contract two tensors (in FP64 or split precision), or evaluate a batch
of tensor networks.  `listed()` names the standing cases, `draw(rng)` gives
further ones of the same ranges, `prepare` / `run` / `exact` make, run and
check one case, and `work` says what one pass cannot do without.

Axis lists are texts: "2^10x48" is ten axes of dim 2, then one of dim 48.
"""
import math
import random

import numpy as np
import torch

from qtnh_amd import _lib, ops

# ---------------------------------------------------------------- the cases


def listed():
    return [
        # A 12-qubit QFT on a resident state, in the order of the reference's
        # example: the smallest whole circuit, bound by latency.
        {"name": "qft_12", "kind": "circuit", "form": "qft", "qubits": 12, "depth": 0, "seed": 0, "readout": False},
        # An ordinary random circuit (SU(2) on every qubit, CZ on a random
        # pairing, from |0...0>), then <Z> on every qubit.
        {"name": "random_20", "kind": "circuit", "form": "random", "qubits": 20, "depth": 10, "seed": 1,
         "readout": True},
        # The same on the largest state the serving workload asks for.
        {"name": "random_28", "kind": "circuit", "form": "random", "qubits": 28, "depth": 6, "seed": 2,
         "readout": True},
        # One gate per call (the reference's one contraction per gate) on a
        # 4 GiB state: dense 1-, 2- and 3-qubit gates and diagonals.
        {"name": "gates_28", "kind": "gates", "rank": 28, "calls": 6, "seed": 3},
        # A full axis permutation of the same state.
        {"name": "permute_28", "kind": "permute", "dims": "2^28", "seed": 4},
        # The same of a tensor whose dims are no powers of two (bond
        # dimensions as they come out of a truncation, spins above 1/2).
        {"name": "permute_ragged", "kind": "permute", "dims": "48x35x81x22x18", "seed": 23},
        # A gate kept as a DenseTensor and contracted into a state with the
        # default placement (its outputs become the last axes).
        {"name": "gate_contract_24", "kind": "contract", "open_a": "2^22", "open_b": "2^2", "wired": "2^2",
         "seed": 6, "gate": True, "split": False},
        # Steps of a network contracted pair by pair: a small one (latency),
        # one of the middle, and one over ragged dims.
        {"name": "step_small", "kind": "contract", "open_a": "2^6", "open_b": "2^5", "wired": "2^5", "seed": 7,
         "gate": False, "split": False},
        {"name": "step_medium", "kind": "contract", "open_a": "2^10", "open_b": "2^10", "wired": "2^9", "seed": 8,
         "gate": False, "split": False},
        {"name": "step_ragged", "kind": "contract", "open_a": "35x29", "open_b": "27x31", "wired": "33x21",
         "seed": 9, "gate": False, "split": False},
        # The largest matrix-like contraction, in split precision.
        {"name": "split_4096", "kind": "contract", "open_a": "4096", "open_b": "4096", "wired": "4096", "seed": 10,
         "gate": False, "split": True},
        # Amplitudes of 4 x 5 grid circuits as tensor networks, contracted
        # together.
        {"name": "networks_32", "kind": "networks", "rows": 4, "cols": 5, "depth": 12, "count": 32, "seed": 11,
         "graph": False},
    ]


def draw(rng):
    kind = rng.choice(["circuit", "circuit", "gates", "permute", "permute", "contract", "contract", "contract",
                       "networks"])
    seed = rng.randrange(1 << 30)
    if kind == "circuit":
        if rng.random() < 0.35:
            return {"kind": kind, "form": "qft", "qubits": rng.randint(6, 24), "depth": 0, "seed": seed,
                    "readout": rng.random() < 0.3}
        return {"kind": kind, "form": "random", "qubits": rng.randint(8, 27), "depth": rng.randint(2, 9),
                "seed": seed, "readout": rng.random() < 0.7}
    if kind == "gates":
        return {"kind": kind, "rank": rng.randint(8, 27), "calls": rng.randint(3, 8), "seed": seed}
    if kind == "permute":
        if rng.random() < 0.5:
            return {"kind": kind, "dims": "2^%d" % rng.randint(8, 28), "seed": seed}
        return {"kind": kind, "dims": _ragged(rng, 2.0 ** rng.uniform(8, 26)), "seed": seed}
    if kind == "contract":
        if rng.random() < 0.3:
            k = rng.randint(1, 3)
            return {"kind": kind, "open_a": "2^%d" % rng.randint(8, 25), "open_b": "2^%d" % k, "wired": "2^%d" % k,
                    "seed": seed, "gate": True, "split": False}
        big = rng.uniform(9, 33)  # log2 of M N K
        parts = [rng.uniform(0.6, 1.4) for _ in range(3)]
        bits = [min(12.5, big * p / sum(parts)) for p in parts]
        if rng.random() < 0.5:
            axes = ["2^%d" % max(1, int(b)) for b in bits]
        else:
            axes = [_ragged(rng, 2.0 ** b) for b in bits]
        return {"kind": kind, "open_a": axes[0], "open_b": axes[1], "wired": axes[2], "seed": seed, "gate": False,
                "split": rng.random() < 0.2}
    return {"kind": kind, "rows": rng.randint(2, 4), "cols": rng.randint(3, 5), "depth": rng.randint(4, 12),
            "count": int(round(2.0 ** rng.uniform(0, 5))), "seed": seed, "graph": rng.random() < 0.3}


def _ragged(rng, size):
    """Axes of dims 2..48 whose product is near `size`."""
    dims, left = [], size
    while left >= 2.0 and len(dims) < 8:
        d = int(round(2.0 ** rng.uniform(1, math.log2(48))))
        if d * 2 > left:
            d = max(2, int(left))
            d = min(d, 48)
        dims.append(d)
        left /= d
    return "x".join(str(d) for d in dims or [2])


def _axes(text):
    out = []
    for part in text.split("x"):
        if "^" in part:
            d, k = part.split("^")
            out += [int(d)] * int(k)
        else:
            out.append(int(part))
    return out


def _size(dims):
    return int(math.prod(dims))


# ------------------------------------------- structure (from the case alone)


def _haar(rng, n):
    g = np.array([complex(rng.gauss(0, 1), rng.gauss(0, 1)) for _ in range(n * n)]).reshape(n, n)
    q, r = np.linalg.qr(g)
    d = np.diagonal(r)
    return q * (d / np.abs(d))


def _phases(rng, n):
    return np.exp(1j * np.array([rng.uniform(0, 2 * math.pi) for _ in range(n)]))


_H = np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2.0)
_CZ = np.array([1, 1, 1, -1], dtype=np.complex128)


def _circuit_ops(case, seed):
    """[(dense?, qubits, coefficients)]; the gates' positions come from the
    case, their values from `seed`."""
    n = case["qubits"]
    out = []
    if case["form"] == "qft":
        for i in range(n):
            out.append((True, [i], _H))
            for j in range(i + 1, n):
                out.append((False, [i, j], np.array([1, 1, 1, np.exp(1j * math.pi / 2 ** (j - i))])))
        return out
    where, values = random.Random(case["seed"]), random.Random("values %d %d" % (case["seed"], seed))
    for _ in range(case["depth"]):
        for q in range(n):
            out.append((True, [q], _haar(values, 2)))
        order = list(range(n))
        where.shuffle(order)
        for p in range(0, n - 1, 2):
            out.append((False, [order[p], order[p + 1]], _CZ))
    return out


def _gate_calls(case, seed):
    n = case["rank"]
    where, values = random.Random(case["seed"]), random.Random("values %d %d" % (case["seed"], seed))
    out = []
    for i in range(case["calls"]):
        dense, k = [(True, 1), (True, 2), (False, 2), (True, 3), (False, 1), (False, 3)][i % 6]
        axes = where.sample(range(n), k)
        out.append((dense, axes, _haar(values, 1 << k) if dense else _phases(values, 1 << k)))
    return out


def _grid_ops(case, which, seed):
    """One grid circuit: SU(2) on every site, then CZ on one of four coupler
    patterns in turn."""
    rows, cols = case["rows"], case["cols"]
    values = random.Random("grid %d %d %d" % (case["seed"], which, seed))
    out = []
    for layer in range(case["depth"]):
        for q in range(rows * cols):
            out.append((True, [q], _haar(values, 2)))
        for r in range(rows):
            for c in range(cols):
                if layer % 4 < 2 and c % 2 == layer % 2 and c + 1 < cols:
                    out.append((False, [r * cols + c, r * cols + c + 1], _CZ))
                if layer % 4 >= 2 and r % 2 == layer % 2 and r + 1 < rows:
                    out.append((False, [r * cols + c, (r + 1) * cols + c], _CZ))
    bits = [values.randrange(2) for _ in range(rows * cols)]
    return out, bits


def _contraction(case):
    """(dims of A, dims of B, wires): A's axes in a mixed order; B's too,
    except that a gate keeps its inputs first, then its outputs."""
    rng = random.Random(case["seed"])
    oa, ob, w = _axes(case["open_a"]), _axes(case["open_b"]), _axes(case["wired"])
    if len(oa) == len(ob) == len(w) == 1:  # plain matrices
        return [oa[0], w[0]], [w[0], ob[0]], [(1, 0)]
    a = [("o", i) for i in range(len(oa))] + [("w", i) for i in range(len(w))]
    b = [("w", i) for i in range(len(w))] + [("o", i) for i in range(len(ob))]
    rng.shuffle(a)
    if not case["gate"]:
        rng.shuffle(b)
    da = [oa[i] if t == "o" else w[i] for t, i in a]
    db = [ob[i] if t == "o" else w[i] for t, i in b]
    return da, db, [(a.index(("w", i)), b.index(("w", i))) for i in range(len(w))]


def _permutation(case):
    dims = _axes(case["dims"])
    ptup = list(range(len(dims)))
    random.Random(case["seed"]).shuffle(ptup)
    return dims, ptup


def _normal(n, gen, scale):
    x = torch.empty(n, dtype=torch.complex128, device="cuda")
    torch.view_as_real(x).normal_(0.0, scale, generator=gen)
    return x


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * case["seed"] + seed)
    kind = case["kind"]
    if kind == "circuit":
        n = 1 << case["qubits"]
        if case["form"] == "qft":
            return _normal(n, gen, math.sqrt(0.5 / n))
        x = torch.zeros(n, dtype=torch.complex128, device="cuda")
        x[0] = 1.0
        return x
    if kind == "gates":
        return _normal(1 << case["rank"], gen, math.sqrt(0.5 / (1 << case["rank"])))
    if kind == "permute":
        return _normal(_size(_axes(case["dims"])), gen, 1.0)
    da, db, _ = _contraction(case)
    return _normal(_size(da), gen, 1.0), _normal(_size(db), gen, 1.0)


def _build(n, ops_list):
    c = ops.Circuit(n)
    for dense, qubits, coef in ops_list:
        (c.gate if dense else c.diag)(qubits, coef)
    return c


def _network(case, which, gates, bits):
    net = ops.Network.amplitude(_build(case["rows"] * case["cols"], gates), bits)
    net.plan_best(seed=case["seed"] + which, max_rank=24, tries=8)
    return net


# ------------------------------------------------------------- one case


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "circuit":
        state["psi"] = _inputs(case, seed)
        state["circuit"] = _build(case["qubits"], _circuit_ops(case, seed))
        state["qubits"] = list(range(case["qubits"]))
    elif kind == "gates":
        state["psi"] = _inputs(case, seed)
        state["dims"] = [2] * case["rank"]
        state["calls"] = _gate_calls(case, seed)
    elif kind == "permute":
        state["x"] = _inputs(case, seed)
        state["dims"], state["ptup"] = _permutation(case)
    elif kind == "contract":
        state["a"], state["b"] = _inputs(case, seed)
        state["da"], state["db"], state["wires"] = _contraction(case)
        state["precision"] = _lib.PREC_SPLIT if case["split"] else _lib.PREC_FP64
    else:
        nets = []
        for i in range(case["count"]):
            gates, bits = _grid_ops(case, i, seed)
            nets.append(_network(case, i, gates, bits))
        state["nets"] = nets
        state["batch"] = ops.NetworkBatch(nets, use_graph=True) if case["graph"] else None
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "circuit":
        psi = state["circuit"].run(state["psi"])
        if state["case"]["readout"]:
            return psi, np.array(ops.expect_z(psi, state["case"]["qubits"], state["qubits"]))
        return psi
    if kind == "gates":
        psi, dims = state["psi"], state["dims"]
        for dense, axes, coef in state["calls"]:
            (ops.gate_apply_ if dense else ops.diag_apply_)(psi, dims, axes, coef)
        return psi
    if kind == "permute":
        return ops.permute(state["x"], state["dims"], state["ptup"])
    if kind == "contract":
        return ops.contract(state["a"], state["da"], state["b"], state["db"], state["wires"],
                            precision=state["precision"])[0]
    if state["batch"] is not None:
        return np.concatenate(state["batch"].run())
    return np.concatenate(ops.run_networks(state["nets"])[0])


def work(case):
    """Bytes: every input and output once (16 per element).  A circuit reads
    and writes its state once however many gates it has; gates applied by one
    call each read and write it once per call.  Flops: 8 per complex
    multiply-add, 6 per complex product."""
    kind = case["kind"]
    if kind in ("circuit", "gates"):
        n = 1 << case["qubits" if kind == "circuit" else "rank"]
        calls = _circuit_ops(case, 0) if kind == "circuit" else _gate_calls(case, 0)
        flops = sum(8 * n * (1 << len(q)) if dense else 6 * n for dense, q, _ in calls)
        if kind == "gates":
            return {"bytes": 32 * n * len(calls), "flops": flops}
        read = 16 * n if case["readout"] else 0
        return {"bytes": 32 * n + read, "flops": flops + (2 * case["qubits"] * n if case["readout"] else 0)}
    if kind == "permute":
        return {"bytes": 32 * _size(_axes(case["dims"])), "flops": 0}
    if kind == "contract":
        m, n, k = (_size(_axes(case[x])) for x in ("open_a", "open_b", "wired"))
        return {"bytes": 16 * (m * k + k * n + m * n), "flops": 8 * m * n * k}
    # Networks: the leaves in (|0>, the gates, the basis state), an amplitude
    # each out; the arithmetic is that of the planned orders.
    sites, leaves, flops = case["rows"] * case["cols"], 0, 0
    for i in range(case["count"]):
        gates, bits = _grid_ops(case, i, 0)
        leaves += 4 * sites + sum(1 << (2 * len(q)) for _, q, _ in gates)
        flops += _network(case, i, gates, bits).info()["flops"]
    return {"bytes": 16 * (leaves + case["count"]), "flops": int(flops)}


# ------------------------------------------------- plain torch, in 64 bits


def _apply(psi, n, dense, qubits, coef):
    """One op on a 2^n vector, out of place for dense ops."""
    order = sorted(qubits)
    shape, last = [], -1
    for q in order:
        shape += [1 << (q - last - 1), 2]
        last = q
    shape.append(1 << (n - 1 - last))
    v = psi.view(shape)
    k = len(qubits)

    def part(t, index):
        where = [slice(None)] * len(shape)
        for m, q in enumerate(qubits):
            where[2 * order.index(q) + 1] = (index >> (k - 1 - m)) & 1
        return t[tuple(where)]

    coef = np.asarray(coef, dtype=np.complex128).reshape(-1)
    if not dense:
        for i in range(1 << k):
            part(v, i).mul_(complex(coef[i]))
        return psi
    out = torch.empty_like(psi)
    w = out.view(shape)
    for o in range(1 << k):
        dst = part(w, o)
        torch.mul(part(v, 0), complex(coef[o]), out=dst)
        for i in range(1, 1 << k):
            dst.add_(part(v, i), alpha=complex(coef[(i << k) + o]))
    return out


def _expect_z(psi, n):
    p = torch.view_as_real(psi).square().sum(dim=1)
    out = []
    for q in range(n):
        halves = p.view(1 << q, 2, -1).sum(dim=(0, 2))
        out.append(float(halves[0] - halves[1]))
    return np.array(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "circuit":
        n, psi = case["qubits"], _inputs(case, seed)
        for dense, qubits, coef in _circuit_ops(case, seed):
            psi = _apply(psi, n, dense, qubits, coef)
        return (psi, _expect_z(psi, n)) if case["readout"] else psi
    if kind == "gates":
        n, psi = case["rank"], _inputs(case, seed)
        for dense, axes, coef in _gate_calls(case, seed):
            psi = _apply(psi, n, dense, axes, coef)
        return psi
    if kind == "permute":
        x = _inputs(case, seed)
        dims, ptup = _permutation(case)
        if set(dims) != {2}:
            back = [0] * len(dims)
            for i, p in enumerate(ptup):
                back[p] = i
            return x.view(dims).permute(back).contiguous().view(-1)
        n = len(dims)
        out = torch.empty_like(x)
        step = min(x.numel(), 1 << 24)
        for lo in range(0, x.numel(), step):
            y = torch.arange(lo, lo + step, dtype=torch.int64, device=x.device)
            src = torch.zeros_like(y)
            for i in range(n):
                src |= ((y >> (n - 1 - ptup[i])) & 1) << (n - 1 - i)
            out[lo:lo + step] = x[src]
        return out
    if kind == "contract":
        a, b = _inputs(case, seed)
        da, db, wires = _contraction(case)
        wa, wb = [w[0] for w in wires], [w[1] for w in wires]
        fa = _as_matrix(a, da, [i for i in range(len(da)) if i not in wa], wa)
        fb = _as_matrix(b, db, wb, [i for i in range(len(db)) if i not in wb])
        return torch.matmul(fa, fb).view(-1)
    n = case["rows"] * case["cols"]
    out = np.zeros(case["count"], dtype=np.complex128)
    for i in range(case["count"]):
        gates, bits = _grid_ops(case, i, seed)
        psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
        psi[0] = 1.0
        for dense, qubits, coef in gates:
            psi = _apply(psi, n, dense, qubits, coef)
        index = 0
        for bit in bits:
            index = 2 * index + bit
        out[i] = complex(psi[index])
    return out


def _as_matrix(x, dims, rows, cols):
    """x as a matrix, its axes `rows` then `cols`.  Many axes: gathered by
    index (torch's copy kernels take fewer axes than a state has)."""
    order = rows + cols
    stride = [_size(dims[i + 1:]) for i in range(len(dims))]
    m = _size([dims[i] for i in rows])
    if len(dims) <= 8:
        return x.view(dims).permute(order).reshape(m, -1)
    rest = torch.arange(x.numel(), dtype=torch.int64, device=x.device)
    src = torch.zeros_like(rest)
    for i in reversed(order):
        src += (rest % dims[i]) * stride[i]
        rest //= dims[i]
    return x[src].view(m, -1)
