"""The work that users of the engine have it do, as cases to measure.

Every case goes through the Python host API (`qiron`): whole circuits on one
state (fresh, repeated and parametric), Trotter steps, SumOp energies and
products, sampling, batches of ansatz energies and the energy surrogate's
training and screening. `listed()` names the cases, `draw()` gives more of the
same ranges, `exact()` restates a case in plain torch with 64-bit numbers.

A state of a case is complex normal and normalised (the amplitudes of a deep
random circuit), written on the device from the seed.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "quant-iron_amd"))

import qiron  # noqa: E402
from qiron import surrogate as S  # noqa: E402


# ---------------------------------------------------------------- the cases --
def listed():
    return [
        # a small circuit, built anew and run on a new state, then its energy: tutorials, unit tests and
        # optimisers of small problems, where launches and allocations count
        dict(name="small_circuit_10q_c128", kind="circuit", n=10, prec="c128", depth=4, fresh=True, energy=True),
        # a one-off run of a 20-qubit circuit (QFT, rotation and CNOT layers) and its energy: planned, run once
        dict(name="qft_energy_20q_c128", kind="qft", n=20, prec="c128", layers=5),
        # one optimiser step of a variational circuit: new angles, the same launch sequence
        dict(name="vqe_step_18q_c64", kind="param", n=18, prec="c64", layers=6),
        # random circuits on mid-size and large states, the plan reused (the second is the benchmark's size)
        dict(name="random_27q_c128", kind="circuit", n=27, prec="c128", depth=10, fresh=False, energy=False),
        dict(name="random_30q_c64", kind="circuit", n=30, prec="c64", depth=40, fresh=False, energy=False),
        # time evolution of a 5 x 5 Heisenberg lattice
        dict(name="trotter_5x5_c64", kind="trotter", rows=5, cols=5, prec="c64", steps=10, order=1),
        # the energy of a chain with fields on a large state
        dict(name="energy_29q_c64", kind="energy", n=29, prec="c64", rows=1),
        # H|psi> of a lattice (Krylov and power methods)
        dict(name="sumop_apply_4x6_c128", kind="apply", n=24, prec="c128", rows=4),
        # 2^18 shots of a 20-qubit register beside 8 others
        dict(name="sample_28q_c64", kind="sample", n=28, prec="c64", measured=20, spread=False, shots=1 << 18),
        # ansatz energies of circuits of uneven sizes with new angles
        dict(name="batch_energies_c64", kind="batch", count=256, nmin=10, nmax=22, prec="c64"),
        # the surrogate: screening of ansatz candidates, and one training epoch
        dict(name="screen_16q6l", kind="screen", count=1 << 19, nang=192, hidden=512),
        dict(name="train_16q6l", kind="train", rows=1 << 14, nang=192, hidden=512, batch=512),
    ]


def draw(rng):
    """One more case: a kind, then sizes over its range."""
    kind = rng.choice(("small", "qft", "param", "circuit", "trotter", "energy", "apply", "sample", "batch", "screen",
                       "train"))
    prec = rng.choice(("c64", "c128"))
    if kind == "small":
        return dict(kind="circuit", n=rng.randint(4, 11), prec=prec, depth=rng.randint(2, 8), fresh=True, energy=prec == "c128")
    if kind == "qft":
        return dict(kind="qft", n=rng.randint(12, 21), prec="c128", layers=rng.randint(1, 5))
    if kind == "param":
        return dict(kind="param", n=rng.randint(12, 24), prec=prec, layers=rng.randint(2, 8))
    if kind == "circuit":
        return dict(kind="circuit", n=rng.randint(14, 28), prec=prec, depth=rng.randint(4, 20), fresh=False, energy=False)
    if kind == "trotter":
        rows, cols = rng.choice(((1, 16), (1, 19), (1, 23), (3, 6), (4, 5), (3, 7), (4, 6), (5, 5)))
        return dict(kind="trotter", rows=rows, cols=cols, prec=prec, steps=rng.randint(1, 10), order=rng.choice((1, 1, 2)))
    if kind == "energy":
        rows = rng.choice((1, 1, 2, 3))
        return dict(kind="energy", n=rows * rng.randint(10 // rows + 1, 28 // rows), prec=prec, rows=rows)
    if kind == "apply":
        rows = rng.choice((1, 2, 3))
        return dict(kind="apply", n=rows * rng.randint(10 // rows + 1, 25 // rows), prec=prec, rows=rows)
    if kind == "sample":
        n = rng.randint(10, 28)
        return dict(kind="sample", n=n, prec=prec, measured=rng.randint(2, min(n, 22)),
                    spread=rng.random() < 0.5, shots=int(2 ** rng.uniform(0, 20)))
    if kind == "batch":
        lo = rng.randint(6, 16)
        return dict(kind="batch", count=int(2 ** rng.uniform(4, 8)), nmin=lo, nmax=rng.randint(lo, 21), prec=prec)
    if kind == "screen":
        return dict(kind="screen", count=int(2 ** rng.uniform(12, 19)), nang=rng.randint(24, 224),
                    hidden=rng.choice((256, 512)))
    return dict(kind="train", rows=int(2 ** rng.uniform(11, 14.5)), nang=rng.randint(24, 224), hidden=rng.choice((256, 512)),
                batch=rng.choice((128, 256, 512, 1024)))


# ------------------------------------------------------- circuits as tuples --
# A gate is (kind, targets, controls, angle); kinds as the engine names them.
ONE_Q = ("H", "X", "Y", "Z", "RX", "RY", "RZ", "P")


def _rng(*key):
    return np.random.default_rng([abs(int(k)) for k in key])


def _random_circuit(n, depth, rng):
    """Per layer a random one-qubit gate on every qubit, n // 2 disjoint CNOT, CZ
    or SWAP pairs and two Toffolis."""
    out = []
    for _ in range(depth):
        for q in range(n):
            k = ONE_Q[rng.integers(8)]
            out.append((k, (q,), (), 2 * math.pi * rng.random() if k in ("RX", "RY", "RZ", "P") else 0.0))
        perm = [int(x) for x in rng.permutation(n)]
        for i in range(n // 2):
            a, b = perm[2 * i], perm[2 * i + 1]
            out.append((("CNOT", (b,), (a,), 0.0), ("Z", (b,), (a,), 0.0), ("SWAP", (a, b), (), 0.0))[rng.integers(3)])
        for _t in range(2):
            a, b, c = (int(x) for x in rng.choice(n, 3, replace=False))
            out.append(("TOFFOLI", (c,), (a, b), 0.0))
    return out


def _qft_circuit(n, layers, rng):
    """QFT on all qubits, then per layer RX, RY, RZ on every qubit and a CNOT ladder."""
    out = []
    for i in range(n):
        out.append(("H", (i,), (), 0.0))
        out += [("P", (i,), (i + k,), math.pi / 2 ** k) for k in range(1, n - i)]
    out += [("SWAP", (i, n - 1 - i), (), 0.0) for i in range(n // 2)]
    for _ in range(layers):
        for kind in ("RX", "RY", "RZ"):
            out += [(kind, (q,), (), 2 * math.pi * rng.random()) for q in range(n)]
        out += [("CNOT", (q + 1,), (q,), 0.0) for q in range(n - 1)]
    return out


def _ansatz(n, angles):
    """Layers of RY and RZ on every qubit and a CNOT ring; angles [layers, 2, n]."""
    out = []
    for a in angles:
        out += [("RY", (q,), (), float(a[0][q])) for q in range(n)]
        out += [("RZ", (q,), (), float(a[1][q])) for q in range(n)]
        out += [("CNOT", ((q + 1) % n,), (q,), 0.0) for q in range(n)]
    return out


def _circuit(n, gates):
    return qiron.Circuit(n, [qiron.Gate.operator(k, t, c, (a,)) for k, t, c, a in gates])


def _lattice(rows, cols, J, h):
    """-1/2 (Jx XX + Jy YY + Jz ZZ) on the open lattice's bonds, -1/2 h Z per site, as ({qubit: 'X'}, coefficient)."""
    out = []
    for s in range(rows * cols):
        out.append(({s: "Z"}, -0.5 * float(h[s])))
        r, c = divmod(s, cols)
        for t in ([s + cols] if r + 1 < rows else []) + ([s + 1] if c + 1 < cols else []):
            out += [({s: p, t: p}, -0.5 * float(j)) for p, j in zip("XYZ", J)]
    return out


def _sumop(terms):
    return qiron.SumOp([qiron.PauliString(c, ops) for ops, c in terms])


def _hamiltonian(rows, cols, rng):
    return _lattice(rows, cols, 0.5 + rng.random(3), 2 * rng.random(rows * cols) - 1)


# ------------------------------------------------------------------- states --
class _Amplitudes:
    """A state's device array (qi_state_device_ptr) for torch; keeps the state alive."""

    def __init__(self, state):
        self.state = state
        n, ptr = state.num_qubits, state.lib.qi_state_device_ptr(state._h)
        self.__cuda_array_interface__ = dict(shape=(1 << n,), typestr="<c16" if state.precision == "c128" else "<c8",
                                             data=(ptr, False), strides=None, version=2)


def _view(state):
    return torch.as_tensor(_Amplitudes(state), device="cuda")


def _fill(v, seed):
    """Complex normal amplitudes of norm 1 from the seed."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    sq = torch.zeros((), dtype=torch.float64, device="cuda")
    parts = torch.view_as_real(v).reshape(-1).split(1 << 27)
    for p in parts:
        p.normal_(generator=g)
        sq += torch.linalg.vector_norm(p, dtype=torch.float64) ** 2
    for p in parts:
        p.mul_((1.0 / sq.sqrt()).to(p.dtype))


def _state(n, prec, seed):
    s = qiron.State.new_zero(n, prec)
    _fill(_view(s), seed)
    torch.cuda.synchronize()  # the engine runs on its own stream
    return s


# ------------------------------------------------------- prepare, run, work --
def _specs(case, seed):
    """The batch's circuits: qubits, layers (the case's) and angles, couplings (the seed's)."""
    shape, rng, out = _rng(case["count"], case["nmin"], case["nmax"]), _rng(seed, 1), []
    for _ in range(case["count"]):
        n, layers = int(shape.integers(case["nmin"], case["nmax"] + 1)), int(shape.integers(4, 9))
        out.append((n, layers, 2 * math.pi * rng.random(2 * n * layers), 0.5 + rng.random(3)))
    return out


def _network(case, seed):
    """Parameters of an n_in -> H -> H -> H -> 1 network (He scale, small biases), in the engine's layout, as a list."""
    rng, H = _rng(seed, 2), case["hidden"]
    n_in = 2 * case["nang"] + 3
    k_in = (n_in + 15) // 16 * 16
    w1 = np.zeros((k_in, H))
    w1[:n_in] = rng.standard_normal((n_in, H)) * math.sqrt(2 / n_in)
    sq = [rng.standard_normal((H, H)) * math.sqrt(2 / H) for _ in range(2)]
    b = [0.1 * rng.standard_normal(H) for _ in range(3)]
    return [a.astype(np.float32) for a in (w1, b[0], sq[0], b[1], sq[1], b[2], rng.standard_normal(H) * math.sqrt(2 / H),
                                           0.1 * rng.standard_normal(1))]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("screen", "train"):
        net = S.MLP(2 * case["nang"] + 3, case["hidden"], seed=1)
        net.set_params(np.concatenate([a.reshape(-1) for a in _network(case, seed)]))
        st = dict(case=case, net=net, seed=int(seed))
        if kind == "train":
            rng = _rng(seed, 3)
            th, J = 2 * math.pi * rng.random((case["rows"], case["nang"])), 0.5 + rng.random((case["rows"], 3))
            t = np.sin(th[:, 0]) * np.cos(th[:, 1]) + J[:, 0] - 1 + 0.1 * rng.standard_normal(case["rows"])
            net.set_data(S.features(th, J), t.astype(np.float32))
        return st
    if kind == "batch":
        specs = _specs(case, seed)
        angles = np.concatenate([s[2] for s in specs])
        return dict(case=case, batch=S.ansatz_batch(specs, case["prec"]), angles=angles)
    if kind == "trotter":
        rows, cols = case["rows"], case["cols"]
        h = _rng(rows, cols).random(rows * cols) - 0.5
        return dict(case=case, terms=_sumop(_lattice(rows, cols, (1.0, 0.8, 1.2), h)).term_array(),
                    state=_state(rows * cols, case["prec"], seed))
    n = case["n"]
    st = dict(case=case, state=_state(n, case["prec"], seed))
    if kind == "circuit":
        gates = _random_circuit(n, case["depth"], _rng(n, case["depth"], seed if case["fresh"] else 0))
        st["circuit"] = _circuit(n, gates)
        st["sumop"] = _sumop(_hamiltonian(1, n, _rng(seed, 4)))
        st["circuit"].array()
    elif kind == "qft":
        st["circuit"] = _circuit(n, _qft_circuit(n, case["layers"], _rng(seed, 5)))
        st["circuit"].array()
        st["sumop"] = _sumop(_hamiltonian(1, n, _rng(seed, 4)))
    elif kind == "param":
        shape = (case["layers"], 2, n)
        gates = _ansatz(n, np.zeros(shape))
        slots, k = [], 0
        for g in gates:
            slots.append(k if g[0] in ("RY", "RZ") else -1)
            k += slots[-1] >= 0
        st["circuit"] = qiron.ParametricCircuit(n, _circuit(n, gates).array(), slots, case["prec"])
        st["angles"] = 2 * math.pi * _rng(seed, 6).random(shape).reshape(-1)
        st["start"], st["state"] = st["state"], qiron.State.new_zero(n, case["prec"])
    elif kind in ("energy", "apply"):
        st["sumop"] = _sumop(_hamiltonian(case["rows"], n // case["rows"], _rng(seed, 4)))
    elif kind == "sample":
        rng = _rng(seed, 7)
        st["qubits"] = list(range(case["measured"]))
        if case["spread"]:
            st["qubits"] = [int(q) for q in np.sort(_rng(n, case["measured"]).permutation(n)[: case["measured"]])]
        st["uniforms"] = rng.random(case["shots"])
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "screen":
        return st["net"].predict_stream(st["seed"], 0, case["count"], case["nang"])
    if kind == "train":
        loss = st["net"].train_epoch(case["batch"], 1e-3, seed=st["seed"])
        return dict(loss=loss, params=st["net"].params())
    if kind == "batch":
        st["batch"].set_angles(st["angles"])
        return st["batch"].run()
    if kind == "trotter":
        qiron.trotter_evolve_terms_inplace(st["state"], st["terms"], 0.02, case["steps"], case["order"])
        return _view(st["state"])
    if kind == "param":
        st["circuit"].set_angles(st["angles"])
        st["state"].copy_from(st["start"])
        return _view(st["circuit"].run(st["state"]))
    if kind == "energy":
        return np.array(st["sumop"].expectation_value(st["state"]))
    if kind == "apply":
        return _view(st["sumop"].apply(st["state"]))
    if kind == "sample":
        return st["state"].measure_outcomes(st["qubits"], st["uniforms"]).astype(np.int64)
    if kind == "circuit" and not case["fresh"]:
        return _view(st["circuit"].execute_inplace(st["state"]))
    out = st["circuit"].execute(st["state"])
    if kind == "circuit" and not case["energy"]:
        return _view(out)
    return [_view(out), np.array(st["sumop"].expectation_value(out))]


def _amp_bytes(case):
    return 16 if case["prec"] == "c128" else 8


def _bonds(rows, cols):
    return rows * (cols - 1) + cols * (rows - 1)


def work(case):
    """What a pass cannot do without: the state (or the network's inputs) read
    and written once, and the arithmetic of the gates, terms or layers."""
    kind = case["kind"]
    if kind in ("screen", "train"):
        n_in, H = 2 * case["nang"] + 3, case["hidden"]
        fwd = 2.0 * (n_in * H + 2 * H * H + H)
        if kind == "screen":
            return dict(bytes=4.0 * case["count"] + 2.0 * (n_in * H + 2 * H * H), flops=fwd * case["count"])
        rows = case["rows"] // case["batch"] * case["batch"]
        return dict(bytes=2.0 * n_in * rows + 24.0 * (n_in * H + 2 * H * H), flops=3 * fwd * rows)
    if kind == "batch":  # states start as |0..0> and end as energies: the angles in, the energies out
        specs = _specs(case, 0)
        ops = sum(2.0 ** n * (layers * n * (8 + 4) + 10 * (n - 1)) for n, layers, _t, _j in specs)
        return dict(bytes=8.0 * sum(s[2].size for s in specs) + 16.0 * len(specs), flops=ops)
    if kind == "trotter":
        n, per = case["rows"] * case["cols"], 3 * _bonds(case["rows"], case["cols"]) + case["rows"] * case["cols"]
        return dict(bytes=2.0 * _amp_bytes(case) * 2 ** n, flops=8.0 * 2 ** n * per * case["steps"] * case["order"])
    n = case["n"]
    size = _amp_bytes(case) * 2.0 ** n
    if kind == "circuit":
        per = n * 7 + n // 2
        return dict(bytes=2 * size, flops=2.0 ** n * per * case["depth"])
    if kind == "qft":
        return dict(bytes=2 * size, flops=2.0 ** n * (n * 4 + n * (n - 1) / 2 * 1.5 + case["layers"] * n * 22 + 10 * n))
    if kind == "param":
        return dict(bytes=2 * size, flops=2.0 ** n * case["layers"] * n * 12)
    if kind == "sample":
        return dict(bytes=size + 24.0 * case["shots"], flops=4.0 * 2 ** n)
    bonds = _bonds(case["rows"], n // case["rows"])
    if kind == "energy":
        return dict(bytes=size, flops=2.0 ** n * (10 * bonds + 4))
    return dict(bytes=2 * size, flops=2.0 ** n * (8 * bonds + 4))


# -------------------------------------------------------- the same in 64 bits --
def _matrix(kind, a):
    c, s = math.cos(a / 2), math.sin(a / 2)
    r = math.sqrt(0.5)
    return {"H": ((r, r), (r, -r)), "X": ((0, 1), (1, 0)), "Y": ((0, -1j), (1j, 0)), "Z": ((1, 0), (0, -1)),
            "RX": ((c, -1j * s), (-1j * s, c)), "RY": ((c, -s), (s, c)),
            "RZ": ((complex(c, -s), 0), (0, complex(c, s))), "P": ((1, 0), (0, complex(math.cos(a), math.sin(a)))),
            "CNOT": ((0, 1), (1, 0)), "TOFFOLI": ((0, 1), (1, 0))}[kind]


def _half(psi, bits):
    """The amplitudes whose qubits have the values of `bits` ({qubit: 0 or 1}), as a view."""
    n, shape, at = psi.numel().bit_length() - 1, [], []
    last = n
    for q in sorted(bits, reverse=True):
        shape += [1 << (last - q - 1), 2]
        at += [slice(None), bits[q]]
        last = q
    return psi.view(*shape, 1 << last)[tuple(at)]


def _gate64(psi, kind, targets, controls, angle):
    on = {c: 1 for c in controls}
    if kind == "SWAP":
        a, b = targets
        x, y = _half(psi, {**on, a: 0, b: 1}), _half(psi, {**on, a: 1, b: 0})
        t = x.clone()
        x.copy_(y)
        y.copy_(t)
        return
    m = _matrix(kind, angle)
    a, b = _half(psi, {**on, targets[0]: 0}), _half(psi, {**on, targets[0]: 1})
    if m[0][1] == 0:
        if m[0][0] != 1:
            a.mul_(m[0][0])
        b.mul_(m[1][1])
        return
    t = a.clone()
    if m[0][0] == 0:
        torch.mul(b, m[0][1], out=a) if m[0][1] != 1 else a.copy_(b)
        torch.mul(t, m[1][0], out=b) if m[1][0] != 1 else b.copy_(t)
        return
    a.mul_(m[0][0]).add_(b, alpha=m[0][1])
    b.mul_(m[1][1]).add_(t, alpha=m[1][0])


def _pauli64(psi, ops):
    out = psi.clone()
    for q, p in ops.items():
        _gate64(out, p, (q,), (), 0.0)
    return out


def _start64(n, prec, seed):
    v = torch.empty(1 << n, dtype=torch.complex128 if prec == "c128" else torch.complex64, device="cuda")
    _fill(v, seed)
    return v.to(torch.complex128)


def _energy64(psi, terms):
    return sum(c * complex(torch.vdot(psi, _pauli64(psi, ops))) for ops, c in terms)


def _uniform64(seed, k):
    """Draws k of the SplitMix64 stream `seed` (Steele, Lea and Flood 2014), 53 bits in [0, 1)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + k.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    return (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _screen64(case, seed):
    w = [torch.from_numpy(a.astype(np.float64)).cuda() for a in _network(case, seed)]
    count, nang, out = case["count"], case["nang"], []
    n_in = 2 * nang + 3
    for c0 in range(0, count, 1 << 16):
        c = np.arange(c0, min(count, c0 + (1 << 16)))
        th = 2 * math.pi * _uniform64(seed, c[:, None] * nang + np.arange(nang) + 1)
        J = 0.5 + _uniform64(seed, count * nang + c[:, None] * 3 + np.arange(3) + 1)
        x = torch.from_numpy(np.concatenate([np.cos(th), np.sin(th), J - 1], axis=1)).cuda()
        for i in range(3):
            x = torch.nn.functional.gelu(x @ w[2 * i][: n_in if i == 0 else None] + w[2 * i + 1])
        out.append(x @ w[6] + w[7])
    return torch.cat(out)


def exact(case, seed):
    """Trained weights and sampled outcomes have no value here, nor has a circuit too large to restate in seconds."""
    kind = case["kind"]
    if kind in ("train", "sample"):
        return None
    if kind == "screen":
        return _screen64(case, int(seed))
    if kind == "batch":
        out = []
        for n, layers, th, J in _specs(case, seed):
            psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
            psi[0] = 1
            for g in _ansatz(n, th.reshape(layers, 2, n)):
                _gate64(psi, *g)
            out.append(_energy64(psi, _lattice(1, n, J, np.zeros(n))))
        return np.array(out)
    if kind == "trotter":
        rows, cols = case["rows"], case["cols"]
        h = _rng(rows, cols).random(rows * cols) - 0.5
        terms = _lattice(rows, cols, (1.0, 0.8, 1.2), h)
        psi = _start64(rows * cols, case["prec"], seed)
        dt = 0.02 / case["order"]
        for _ in range(case["steps"]):
            for ops, c in terms + (terms[::-1] if case["order"] == 2 else []):
                psi = math.cos(dt * c) * psi + complex(0, -math.sin(dt * c)) * _pauli64(psi, ops)
        return psi
    n = case["n"]
    if kind == "circuit":
        gates = _random_circuit(n, case["depth"], _rng(n, case["depth"], seed if case["fresh"] else 0))
    elif kind == "qft":
        gates = _qft_circuit(n, case["layers"], _rng(seed, 5))
    elif kind == "param":
        gates = _ansatz(n, 2 * math.pi * _rng(seed, 6).random((case["layers"], 2, n)))
    else:
        terms = _hamiltonian(case["rows"], n // case["rows"], _rng(seed, 4))
        psi = _start64(n, case["prec"], seed)
        if kind == "energy":
            return np.array(_energy64(psi, terms))
        out = torch.zeros_like(psi)
        for ops, c in terms:
            out += c * _pauli64(psi, ops)
        return out
    if len(gates) * 2.0 ** n > 2.0 ** 37:
        return None
    psi = _start64(n, case["prec"], seed)
    for g in gates:
        _gate64(psi, *g)
    if kind == "param" or not (kind == "qft" or case["energy"]):
        return psi
    return [psi, np.array(_energy64(psi, _hamiltonian(1, n, _rng(seed, 4))))]
