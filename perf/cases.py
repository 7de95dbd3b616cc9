"""Performance cases: the work that a user of this framework has it do.

A case is a dict of plain values; ``prepare`` builds what a program holds
before the call (states, circuits, engines), ``run`` makes one pass through
the public entry points.  Circuits are written as plain (gate, qubits,
parameters) lists, so that ``prepare`` can turn them into gate objects and
``exact`` can evolve them with dense matrices in 64 bits.  The gate structure
of a case follows from the case alone; parameters and states follow from the
seed.
"""

import math
import random

import numpy as np
import torch

from qibojit_amd._qibo import Circuit, gates
from qibojit_amd.ansatz import AnsatzEnergy, AnsatzEngine, HardwareEfficientAnsatz
from qibojit_amd.backends import clifford_operations_hip as clifford
from qibojit_amd.backends.hip import HipBackend
from qibojit_amd.batch import AnsatzBatch
from qibojit_amd.fusion import fuse_blocks

DEVICE = "cuda"
TORCH_TYPES = {"complex64": torch.complex64, "complex128": torch.complex128}
AMP_BYTES = {"complex64": 8, "complex128": 16}
METROPOLIS_CHAINS = 16


def listed():
    return [
        # A short program on a few qubits, one call per gate: latency and
        # launches, no memory traffic to speak of.
        {"name": "gates_10q", "kind": "gates", "n": 10, "dtype": "complex128", "ngates": 48, "structure": 1},
        # The gate sweep of bench.py at its size: every gate family on the
        # first, middle and last qubit of a 30-qubit double-precision state.
        {"name": "sweep_30q", "kind": "sweep", "n": 30, "dtype": "complex128"},
        # bench.py's random circuit: a cache-resident state, fused execution.
        {"name": "random_20q", "kind": "random", "n": 20, "dtype": "complex128", "depth": 20, "structure": 3},
        # Quantum Fourier transform in single precision, fused execution of
        # a state far beyond the caches.
        {"name": "qft_30q", "kind": "qft", "n": 30, "dtype": "complex64"},
        # Brickwork of random two-qubit unitaries, fused into dense blocks of
        # up to five qubits (an odd number of qubits, no power-of-two layers).
        {"name": "brickwork_27q", "kind": "blocks", "n": 27, "dtype": "complex64", "depth": 6},
        # Noisy circuit on a density matrix: gates, Pauli noise on every qubit
        # after each layer, amplitude damping at the end.
        {"name": "noisy_density_12q", "kind": "density", "n": 12, "dtype": "complex128", "depth": 2},
        # Measuring a large state: marginal probabilities, shots, collapse.
        {"name": "measure_28q", "kind": "measure", "n": 28, "dtype": "complex128", "measured": 10, "nshots": 20000,
         "structure": 7},
        # One energy evaluation of a variational program: run the ansatz as a
        # circuit, then the transverse-field Ising expectation of its state.
        {"name": "energy_26q", "kind": "energy", "n": 26, "dtype": "complex128", "layers": 2},
        # Training step of a batch of parameter sets: energies and the
        # gradients of every parameter through autograd.
        {"name": "gradient_22q", "kind": "gradient", "n": 22, "dtype": "complex64", "layers": 6, "batch": 16},
        # Many ansatz circuits of uneven shape with new parameters on each
        # step, replayed as one graph.
        {"name": "batch_192", "kind": "batch", "circuits": 192, "nmin": 8, "nmax": 20, "dtype": "complex64",
         "structure": 11},
        # Stabilizer simulation of a wide circuit: a random Clifford gate
        # list and a collapsing measurement of every qubit.
        {"name": "clifford_1000q", "kind": "clifford", "n": 1000, "ngates": 20000},
        # Many shots of a stabilizer state.
        {"name": "clifford_shots_100q", "kind": "shots", "n": 100, "measured": 100, "nshots": 10000},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["gates", "sweep", "random", "qft", "blocks", "density", "measure", "energy", "gradient",
                       "batch", "clifford", "shots"])
    dtype = rng.choice(["complex64", "complex128"])
    structure = rng.randrange(1, 1 << 20)
    if kind == "gates":
        return {"kind": kind, "n": rng.randint(4, 28), "dtype": dtype, "ngates": rng.randint(8, 48),
                "structure": structure}
    if kind == "sweep":
        return {"kind": kind, "n": rng.randint(8, 29), "dtype": dtype}
    if kind == "random":
        return {"kind": kind, "n": rng.randint(5, 25), "dtype": dtype, "depth": rng.randint(3, 20),
                "structure": structure}
    if kind == "qft":
        return {"kind": kind, "n": rng.randint(6, 29), "dtype": dtype}
    if kind == "blocks":
        return {"kind": kind, "n": rng.randint(10, 26), "dtype": dtype, "depth": rng.randint(3, 8)}
    if kind == "density":
        return {"kind": kind, "n": rng.randint(3, 12), "dtype": dtype, "depth": rng.randint(1, 2)}
    if kind == "measure":
        n = rng.randint(11, 28)
        return {"kind": kind, "n": n, "dtype": "complex128", "measured": rng.randint(1, min(n, 16)),
                "nshots": _log_int(rng, 100, 400000), "structure": structure}
    if kind == "energy":
        return {"kind": kind, "n": rng.randint(6, 26), "dtype": dtype, "layers": rng.randint(1, 3)}
    if kind == "gradient":
        return {"kind": kind, "n": rng.randint(6, 22), "dtype": dtype, "layers": rng.randint(2, 6),
                "batch": rng.randint(1, 16)}
    if kind == "batch":
        nmin = rng.randint(6, 12)
        return {"kind": kind, "circuits": _log_int(rng, 16, 192), "nmin": nmin, "nmax": rng.randint(nmin, 19),
                "dtype": dtype, "structure": structure}
    if kind == "clifford":
        return {"kind": kind, "n": _log_int(rng, 20, 1200), "ngates": _log_int(rng, 500, 20000)}
    n = _log_int(rng, 10, 150)
    return {"kind": kind, "n": n, "measured": rng.randint(1, n), "nshots": _log_int(rng, 100, 20000)}


# ------------------------------------------------------------- circuits --
def _haar(rng, dim):
    z = (rng.standard_normal((dim, dim)) + 1j * rng.standard_normal((dim, dim))) / np.sqrt(2)
    q, r = np.linalg.qr(z)
    return q * (np.diag(r) / np.abs(np.diag(r)))


# gate -> (qubits, angles, share of the amplitudes it can change)
FAMILIES = {
    "H": (1, 0, 1.0), "X": (1, 0, 1.0), "Z": (1, 0, 0.5), "RY": (1, 1, 1.0), "RZ": (1, 1, 1.0), "U3": (1, 3, 1.0),
    "CNOT": (2, 0, 0.5), "CZ": (2, 0, 0.25), "CU1": (2, 1, 0.25), "CU3": (2, 3, 0.5), "SWAP": (2, 0, 0.5),
    "fSim": (2, 2, 0.75), "TOFFOLI": (3, 0, 0.25), "Unitary2": (2, 0, 1.0), "Unitary3": (3, 0, 1.0),
}
CONTROLS = {"CNOT": 1, "CZ": 1, "CU1": 1, "CU3": 1, "TOFFOLI": 2}


def _specs(case, seed):
    """The case's gates as (name, qubits, parameters)."""
    n, kind = case["n"], case["kind"]
    rng = np.random.default_rng(seed)
    shape = random.Random(case.get("structure", 0))
    out = []

    def add(name, *qubits):
        if name.startswith("Unitary"):
            params = (_haar(rng, 2 ** len(qubits)),)
        else:
            params = tuple(float(x) for x in rng.uniform(-np.pi, np.pi, FAMILIES[name][1]))
        out.append((name, qubits, params))

    if kind == "gates":
        names = sorted(FAMILIES)
        for _ in range(case["ngates"]):
            name = shape.choice(names)
            add(name, *shape.sample(range(n), FAMILIES[name][0]))
    elif kind == "sweep":
        for t in (0, n // 2, n - 1):
            pair = (t, t + 1) if t < n - 1 else (t - 1, t)
            ctrl = t + 1 if t < n - 1 else t - 1
            three = (t, t + 1, t + 2) if t + 2 < n else (n - 3, n - 2, n - 1)
            for name in ("H", "X", "Z", "RZ"):
                add(name, t)
            add("CNOT", ctrl, t)
            add("SWAP", *pair)
            add("fSim", *pair)
            add("CU3", ctrl, t)
            add("Unitary3", *three)
    elif kind == "random":
        for _ in range(case["depth"]):
            for q in range(n):
                add("U3", q)
            order = list(range(n))
            shape.shuffle(order)
            for a, b in zip(order[0::2], order[1::2]):
                add("CZ", a, b)
    elif kind == "qft":
        for i in range(n):
            out.append(("H", (i,), ()))
            for j in range(i + 1, n):
                out.append(("CU1", (j, i), (math.pi / 2 ** (j - i),)))
        for i in range(n // 2):
            out.append(("SWAP", (i, n - i - 1), ()))
    elif kind == "blocks":
        for layer in range(case["depth"]):
            for q in range(layer % 2, n - 1, 2):
                add("Unitary2", q, q + 1)
    elif kind == "density":
        for layer in range(case["depth"]):
            for q in range(n):
                add("U3", q)
            for q in range(layer % 2, n - 1, 2):
                add("CNOT", q, q + 1)
            for q in range(n):
                out.append(("pauli", (q,), tuple(float(x) for x in rng.uniform(0.0, 0.02, 3))))
        for q in range(0, n, 3):
            out.append(("damping", (q,), (float(rng.uniform(0.01, 0.1)),)))
    return out


PAULIS = (np.array([[0, 1], [1, 0]], dtype=complex), np.array([[0, -1j], [1j, 0]]), np.diag([1, -1]).astype(complex))


def _damping(gamma):
    return (np.array([[1, 0], [0, math.sqrt(1 - gamma)]], dtype=complex),
            np.array([[0, math.sqrt(gamma)], [0, 0]], dtype=complex))


def _gate(name, qubits, params):
    if name.startswith("Unitary"):
        return gates.Unitary(params[0], *qubits)
    if name == "pauli":
        return gates.UnitaryChannel([qubits] * 3, list(zip(params, PAULIS)))
    if name == "damping":
        return gates.KrausChannel([qubits] * 2, list(_damping(*params)))
    return getattr(gates, name)(*qubits, *params)


def _circuit(case, seed, density=False):
    circuit = Circuit(case["n"], density_matrix=density)
    for spec in _specs(case, seed):
        circuit.add(_gate(*spec))
    return circuit


# --------------------------------------------------------------- inputs --
def _normals(seed, shape, tdtype):
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    return torch.randn(shape, dtype=tdtype, device=DEVICE, generator=gen)


def _state(case, seed):
    """A random pure state (amplitudes as of a deep circuit)."""
    state = _normals(seed, (1 << case["n"],), TORCH_TYPES[case["dtype"]])
    state /= torch.linalg.vector_norm(state)
    return state


def _density(case, seed):
    """A mixture of two random pure states."""
    dim = 1 << case["n"]
    a = _normals(seed, (2, dim), torch.complex128)
    a /= torch.linalg.vector_norm(a, dim=1, keepdim=True)
    rho = 0.75 * torch.outer(a[0], a[0].conj()) + 0.25 * torch.outer(a[1], a[1].conj())
    return rho.to(TORCH_TYPES[case["dtype"]])


def _backend(case):
    backend = HipBackend()
    backend.set_dtype(case["dtype"])
    return backend


def _measurement(case, seed):
    """(measured qubits, qubits to collapse, outcome)."""
    shape = random.Random(case["structure"])
    measured = sorted(shape.sample(range(case["n"]), case["measured"]))
    collapsed = measured[: min(3, len(measured))]
    return measured, collapsed, int(np.random.default_rng(seed).integers(2 ** len(collapsed)))


def _angles(case, seed, batch=None):
    ansatz = HardwareEfficientAnsatz(case["n"], case["layers"])
    return ansatz, ansatz.random_parameters(np.random.default_rng(seed), batch)


def _batch_shapes(case):
    shape = random.Random(case["structure"])
    return [(shape.randint(case["nmin"], case["nmax"]), shape.randint(2, 10)) for _ in range(case["circuits"])]


def _batch_params(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(-np.pi, np.pi, 2 * n * layers) for n, layers in _batch_shapes(case)]


def _clifford_gates(n, ngates, seed):
    """Random gate list in the engine's (kind, q0, q1) rows, 40% two-qubit."""
    rng = np.random.default_rng(seed)
    one = [k for name, k in clifford.KINDS.items() if name not in clifford.TWO_QUBIT]
    two = [clifford.KINDS[name] for name in clifford.TWO_QUBIT]
    q0 = rng.integers(n, size=ngates)
    q1 = (q0 + 1 + rng.integers(n - 1, size=ngates)) % n
    pick = rng.random(ngates) < 0.4
    kinds = np.where(pick, rng.choice(two, ngates), rng.choice(one, ngates))
    return np.ascontiguousarray(np.stack([kinds, q0, np.where(pick, q1, -1)], axis=1).astype(np.int32))


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "n": case.get("n")}
    if kind in ("gates", "sweep"):
        s.update(backend=_backend(case), gates=[_gate(*spec) for spec in _specs(case, seed)], state=_state(case, seed))
    elif kind in ("random", "qft"):
        s.update(backend=_backend(case), circuit=_circuit(case, seed), state=_state(case, seed))
    elif kind == "blocks":
        s.update(backend=_backend(case), gates=list(fuse_blocks(_circuit(case, seed), 5).queue),
                 state=_state(case, seed))
    elif kind == "density":
        s.update(backend=_backend(case), circuit=_circuit(case, seed, True), state=_density(case, seed))
    elif kind == "measure":
        backend = _backend(case)
        backend.set_seed(seed)
        backend.set_threads(METROPOLIS_CHAINS)
        measured, collapsed, outcome = _measurement(case, seed)
        s.update(backend=backend, state=_state(case, seed), measured=measured, collapsed=collapsed, outcome=outcome,
                 nshots=case["nshots"])
    elif kind == "energy":
        ansatz, params = _angles(case, seed)
        s.update(backend=_backend(case), circuit=ansatz.circuit(params))
    elif kind == "gradient":
        ansatz, params = _angles(case, seed, case["batch"])
        s.update(engine=AnsatzEngine(ansatz, case["batch"], dtype=case["dtype"]),
                 params=torch.tensor(params, dtype=torch.float64, device=DEVICE, requires_grad=True))
    elif kind == "batch":
        batch = AnsatzBatch(_batch_shapes(case), dtype=case["dtype"])
        params = _batch_params(case, seed)
        batch.set_parameters(params)
        batch.capture()
        s.update(batch=batch, params=params)
    elif kind == "clifford":
        n = case["n"]
        np.random.seed(seed % (1 << 32))
        s.update(tableau=clifford.zero_state(n), gates=_clifford_gates(n, case["ngates"], seed))
    else:
        n = case["n"]
        np.random.seed(seed % (1 << 32))
        tableau = clifford.apply_circuit(clifford.zero_state(n), _clifford_gates(n, 20 * n, seed), n)
        s.update(tableau=tableau, qubits=list(range(case["measured"])), nshots=case["nshots"])
    return s


def run(s):
    kind, n = s["kind"], s["n"]
    if kind in ("gates", "sweep", "blocks"):
        backend, state = s["backend"], s["state"]
        for gate in s["gates"]:
            state = backend.apply_gate(gate, state, n)
        return state
    if kind in ("random", "qft", "density"):
        return s["backend"].execute_circuit(s["circuit"], initial_state=s["state"]).state()
    if kind == "measure":
        backend = s["backend"]
        probs = backend.calculate_probabilities(s["state"], s["measured"], n)
        counts = backend.sample_frequencies(probs, s["nshots"])
        histogram = np.zeros(len(probs), dtype=np.int64)
        histogram[list(counts.keys())] = list(counts.values())
        state = backend.collapse_state(s["state"], s["collapsed"], s["outcome"], n)
        return probs, histogram, state
    if kind == "energy":
        backend = s["backend"]
        state = backend.execute_circuit(s["circuit"]).state()
        return state, backend.expectation_tfim(state, n)
    if kind == "gradient":
        energies = AnsatzEnergy.apply(s["params"], s["engine"])
        (gradients,) = torch.autograd.grad(energies.sum(), s["params"])
        return energies.detach(), gradients
    if kind == "batch":
        batch = s["batch"]
        batch.set_parameters(s["params"])
        batch.replay()
        return batch.energies()
    if kind == "clifford":
        tableau = clifford.apply_circuit(s["tableau"], s["gates"], n)
        outcomes = clifford.M(tableau, range(n), n, collapse=True)
        return np.array(outcomes, dtype=np.int64), clifford._clifford_post_execution_reshape(tableau, n)
    return clifford.sample_shots(s["tableau"], s["qubits"], n, s["nshots"])


def work(case):
    kind = case["kind"]
    if kind in ("clifford", "shots"):
        tableau = (2 * case["n"] + 1) ** 2 / 8
        extra = case["nshots"] * case["measured"] if kind == "shots" else (2 * case["n"] + 1) ** 2
        steps = case["ngates"] if kind == "clifford" else case["measured"]
        return {"bytes": 2 * tableau + extra, "flops": steps * (2 * case["n"] + 1) / 8}
    if kind == "batch":
        shapes = _batch_shapes(case)
        return {"bytes": sum(2 * n * layers * 8 + 8 for n, layers in shapes),
                "flops": sum(2.0**n * layers * n * 16 for n, layers in shapes)}
    n = case["n"]
    amps = float(1 << n)
    amp = AMP_BYTES[case["dtype"]]
    if kind in ("gates", "sweep"):  # separate calls: each reads and writes what its gate can change
        share = [FAMILIES[name][2] for name, _, _ in _specs(case, 0)]
        size = [len(q) - CONTROLS.get(name, 0) for name, q, _ in _specs(case, 0)]
        return {"bytes": 2 * amp * amps * sum(share), "flops": amps * sum(f * 8 * 2**k for f, k in zip(share, size))}
    if kind == "blocks":
        nblocks = len(fuse_blocks(_circuit(case, 0), 5).queue)
        return {"bytes": 2 * amp * amps * nblocks, "flops": amps * 8 * 4 * len(_specs(case, 0))}
    if kind in ("random", "qft"):
        flops = sum(FAMILIES[name][2] * 8 * 2 ** (len(q) - CONTROLS.get(name, 0)) for name, q, _ in _specs(case, 0))
        return {"bytes": 2 * amp * amps, "flops": amps * flops}
    if kind == "density":
        return {"bytes": 2 * amp * amps * amps, "flops": amps * amps * 32 * len(_specs(case, 0))}
    if kind == "measure":
        kept = 0.5 ** min(3, case["measured"])
        return {"bytes": amp * amps * (1 + 1 + kept), "flops": amps * 8}
    if kind == "energy":
        return {"bytes": 2 * amp * amps, "flops": amps * (case["layers"] * 40 * n + 4 * n)}
    # gradient: parameters in, energies and gradients out
    count = case["batch"] * 2 * n * case["layers"]
    return {"bytes": 16.0 * count, "flops": amps * case["batch"] * n * (case["layers"] * (16 + 2 * 32) + 4)}


# -------------------------------------------------------- 64-bit results --
def _matrix(name, params):
    """(matrix over the targets, number of leading control qubits)."""
    e, c, s = np.exp, np.cos, np.sin
    nc = CONTROLS.get(name, 0)
    if name == "H":
        return np.array([[1, 1], [1, -1]], dtype=complex) / math.sqrt(2), nc
    if name in ("X", "CNOT", "TOFFOLI"):
        return PAULIS[0], nc
    if name in ("Z", "CZ"):
        return PAULIS[2], nc
    if name == "CU1":
        return np.diag([1, e(1j * params[0])]), nc
    if name == "RY":
        t = params[0] / 2
        return np.array([[c(t), -s(t)], [s(t), c(t)]], dtype=complex), nc
    if name == "RZ":
        return np.diag([e(-0.5j * params[0]), e(0.5j * params[0])]), nc
    if name in ("U3", "CU3"):
        t, p, m = params[0] / 2, (params[1] + params[2]) / 2, (params[1] - params[2]) / 2
        return np.array([[e(-1j * p) * c(t), -e(-1j * m) * s(t)], [e(1j * m) * s(t), e(1j * p) * c(t)]]), nc
    if name == "SWAP":
        return np.eye(4, dtype=complex)[[0, 2, 1, 3]], nc
    if name == "fSim":
        t, p = params
        return np.array([[1, 0, 0, 0], [0, c(t), -1j * s(t), 0], [0, -1j * s(t), c(t), 0], [0, 0, 0, e(-1j * p)]]), nc
    return np.asarray(params[0], dtype=complex), nc


def _evolve(state, nbits, matrix, targets, controls=()):
    """Dense gate on a flat state, in place, by slices (qubit 0 = top bit)."""
    every = sorted([*targets, *controls])
    dims, last = [], -1
    for q in every:
        dims += [1 << (q - last - 1), 2]
        last = q
    view = state.view(*dims, 1 << (nbits - last - 1))
    axis = {q: 2 * i + 1 for i, q in enumerate(every)}
    parts = []
    for r in range(2 ** len(targets)):
        index = [slice(None)] * view.dim()
        for q in controls:
            index[axis[q]] = 1
        for i, q in enumerate(targets):
            index[axis[q]] = (r >> (len(targets) - 1 - i)) & 1
        parts.append(view[tuple(index)])
    new = []
    for row in matrix:
        total = None
        for value, part in zip(row, parts):
            if value != 0:
                term = part * complex(value)
                total = term if total is None else total.add_(term)
        new.append(torch.zeros_like(parts[0]) if total is None else total)
    for part, value in zip(parts, new):
        part.copy_(value)
    return state


def _evolve_specs(state, nbits, specs):
    for name, qubits, params in specs:
        matrix, nc = _matrix(name, params)
        _evolve(state, nbits, matrix, qubits[nc:], qubits[:nc])
    return state


def _evolve_density(rho, n, specs):
    flat = rho.reshape(-1)

    def conjugate(x, m, targets, controls=()):
        _evolve(x, 2 * n, m, targets, controls)
        return _evolve(x, 2 * n, m.conj(), [q + n for q in targets], [q + n for q in controls])

    for name, qubits, params in specs:
        if name == "pauli":
            new = flat * (1 - sum(params))
            for p, m in zip(params, PAULIS):
                new += p * conjugate(flat.clone(), m, qubits)
            flat = new
        elif name == "damping":
            flat = sum(conjugate(flat.clone(), m, qubits) for m in _damping(*params))
        else:
            m, nc = _matrix(name, params)
            conjugate(flat, m, qubits[nc:], qubits[:nc])
    return flat.reshape(rho.shape)


def _rotate(psi, n, q, m00, m01, m10, m11):
    """One-qubit matrices, one per row of a batch of states, in place."""
    view = psi.view(psi.shape[0], 1 << q, 2, -1)
    a, b = view[:, :, 0], view[:, :, 1]
    m00, m01, m10, m11 = (torch.as_tensor(m, dtype=torch.complex128, device=DEVICE).view(-1, 1, 1)
                          for m in (m00, m01, m10, m11))
    new = a * m00 + b * m01
    b.copy_(a * m10 + b * m11)
    a.copy_(new)


def _ising(psi, n, g=1.0):
    """H psi of -sum Z Z - g sum X for a batch of states."""
    k = torch.arange(1 << n, device=DEVICE)
    flips = (k ^ (k >> 1)) & ((1 << (n - 1)) - 1)
    diagonal = torch.full((1 << n,), -(n - 1.0), dtype=torch.float64, device=DEVICE)
    for i in range(n - 1):
        diagonal += 2.0 * ((flips >> i) & 1)
    out = psi * diagonal
    for q in range(n):
        out -= g * psi.view(psi.shape[0], 1 << q, 2, -1).flip(2).reshape(psi.shape)
    return out


def _ansatz_states(n, layers, params):
    """States of a batch of ansatz circuits (RY, RZ, CNOT ladder per layer)."""
    batch = params.shape[0]
    angles = params.reshape(batch, layers, 2, n)
    psi = torch.zeros((batch, 1 << n), dtype=torch.complex128, device=DEVICE)
    psi[:, 0] = 1
    k = torch.arange(1 << n, device=DEVICE)
    gather = k ^ (k >> 1)
    for layer in range(layers):
        c, s = np.cos(angles[:, layer, 0] / 2), np.sin(angles[:, layer, 0] / 2)
        z = np.exp(-0.5j * angles[:, layer, 1])
        for q in range(n):
            zq, cq, sq = z[:, q], c[:, q], s[:, q]
            _rotate(psi, n, q, zq * cq, -zq * sq, zq.conj() * sq, zq.conj() * cq)
        psi = psi[:, gather]
    return psi


def _ansatz_gradients(n, layers, params):
    batch = params.shape[0]
    angles = params.reshape(batch, layers, 2, n)
    psi = _ansatz_states(n, layers, params)
    lam = _ising(psi, n)
    energies = (psi.conj() * lam).sum(dim=1).real
    grads = torch.empty((batch, layers, 2, n), dtype=torch.float64, device=DEVICE)
    k = torch.arange(1 << n, device=DEVICE)
    gather = k ^ (k >> 1)
    undo = torch.empty_like(gather)
    undo[gather] = k
    for layer in reversed(range(layers)):
        psi, lam = psi[:, undo], lam[:, undo]
        for q in range(n):
            t, p = angles[:, layer, 0, q] / 2, angles[:, layer, 1, q]
            v, w = psi.view(batch, 1 << q, 2, -1), lam.view(batch, 1 << q, 2, -1)
            grads[:, layer, 1, q] = ((w[:, :, 0].conj() * v[:, :, 0]).sum(dim=(1, 2))
                                     - (w[:, :, 1].conj() * v[:, :, 1]).sum(dim=(1, 2))).imag
            e = np.exp(0.5j * p)
            for x in (psi, lam):
                _rotate(x, n, q, e, 0 * e, 0 * e, e.conj())
            grads[:, layer, 0, q] = (-1j * (w[:, :, 0].conj() * v[:, :, 1]).sum(dim=(1, 2))
                                     + 1j * (w[:, :, 1].conj() * v[:, :, 0]).sum(dim=(1, 2))).imag
            for x in (psi, lam):
                _rotate(x, n, q, np.cos(t), np.sin(t), -np.sin(t), np.cos(t))
    return energies, grads.reshape(batch, -1)


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind in ("gates", "sweep", "blocks", "random", "qft"):
        return _evolve_specs(_state(case, seed).to(torch.complex128), n, _specs(case, seed))
    if kind == "density":
        return _evolve_density(_density(case, seed).to(torch.complex128), n, _specs(case, seed))
    if kind == "measure":
        measured, collapsed, outcome = _measurement(case, seed)
        state = _state(case, seed)
        dims, last = [], -1
        for q in measured:
            dims += [1 << (q - last - 1), 2]
            last = q
        squares = (state.real.square() + state.imag.square()).view(*dims, -1)
        probs = squares
        for axis in range(2 * len(measured), -1, -2):
            probs = probs.sum(dim=axis)
        probs = probs.reshape(-1)
        keep = torch.zeros_like(squares, dtype=torch.bool)
        index = [slice(None)] * squares.dim()
        for i in range(len(collapsed)):
            index[2 * i + 1] = (outcome >> (len(collapsed) - 1 - i)) & 1
        keep[tuple(index)] = True
        state = torch.where(keep.view(-1), state, torch.zeros_like(state))
        return probs, None, state / torch.linalg.vector_norm(state)
    if kind == "energy":
        ansatz, params = _angles(case, seed)
        psi = _ansatz_states(n, ansatz.nlayers, params.reshape(1, -1))
        energy = float((psi.conj() * _ising(psi, n)).sum().real)
        return psi.reshape(-1), energy
    if kind == "gradient":
        return _ansatz_gradients(n, case["layers"], _angles(case, seed, case["batch"])[1])
    if kind == "batch":
        out = []
        for (m, layers), params in zip(_batch_shapes(case), _batch_params(case, seed)):
            psi = _ansatz_states(m, layers, params.reshape(1, -1))
            out.append((psi.conj() * _ising(psi, m)).sum().real)
        return torch.stack(out)
    return None  # stabilizer tableaux and samples are whole numbers
