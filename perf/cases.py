"""The measured work of the statevector engine: what its users call, at the sizes they call it.

Every case is one call (or the short fixed sequence of calls one program step makes) through the
package's public entry points. Families and what they stand for in use:

  simulate    quafu-style `simulate(qc, shots, hamiltonian)` on a handful of qubits: state, counts and
              expectations back on the host; latency and launches count
  circuit     a layered random circuit (U3 on every qubit, CX brickwork, CRZ on random pairs) on a
              device state: small registers read back whole, large ones through the amplitudes of
              given bitstrings (cross-entropy benchmarking) and the expectations of a Hamiltonian, as a
              program with a state of gigabytes does
  qft         the textbook QFT of a basis state and the Bloch vector of every qubit (phase estimation's
              inner routine: controlled phases on every pair)
  two_target  circuits of gates with dense two-qubit matrices (SWAP, iSWAP, RXX, RYY, controlled SWAP)
  blocks      deep circuits confined to blocks of a few qubits (unitary blocks on 4 or 5 qubits)
  adjoint     one training step of a hardware-efficient ansatz: loss and every gradient through the
              torch layer
  batch       one training step over many ansatz circuits of uneven sizes
  sample      shots from a state that is already on the device
  expect      the energy terms of a Hamiltonian on a state that is already on the device
  noisy       trajectories of a circuit with depolarizing and damping channels

Circuits are lists of (name, qubits, angles), from which both the package's circuit and the plain
64-bit evaluation (`exact`) are made.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import pyquafu_amd as pq
from pyquafu_amd import _native
from pyquafu_amd.algorithms.hamiltonian import Hamiltonian, PauliOp
from pyquafu_amd.algorithms.interface.torch import expectation
from pyquafu_amd.batch import BatchRunner, compile_item
from pyquafu_amd.elements import (AmplitudeDamping, CPGate, CRZGate, CSwapGate, CXGate, CZGate, Depolarizing, HGate,
                                  ISwapGate, Parameter, RXXGate, RYGate, RYYGate, RZGate, SwapGate, U3Gate, XGate)
from pyquafu_amd.simulators import simulate
from pyquafu_amd.simulators.program import compile_circuit

# ------------------------------------------------------------------------------------------------ cases


def listed():
    return [
        # the smallest whole call: the smoke test's circuit with shots and <Z_i>
        {"name": "simulate_12q", "family": "simulate", "n": 12, "layers": 6, "crz": 3, "shots": 100, "dtype": "c128"},
        # the CPU-parity workload: 20 qubits, depth 20, state read back
        {"name": "circuit_20q_c128", "family": "circuit", "n": 20, "layers": 20, "crz": 0, "dtype": "c128"},
        # the headline workload's register (16 GiB), ten of its layers, energy read out
        {"name": "circuit_30q_c128", "family": "circuit", "n": 30, "layers": 10, "crz": 15, "dtype": "c128"},
        # single precision on an odd register
        {"name": "circuit_27q_c64", "family": "circuit", "n": 27, "layers": 8, "crz": 13, "dtype": "c64"},
        # the QFT workload at a register that leaves room for a second state
        {"name": "qft_28q_c128", "family": "qft", "n": 28, "dtype": "c128"},
        # dense two-qubit gates in single precision
        {"name": "two_target_25q_c64", "family": "two_target", "n": 25, "layers": 8, "dtype": "c64"},
        # deep five-qubit blocks; 27 = 5 * 5 + 2 leaves a short last block
        {"name": "blocks_27q_c128", "family": "blocks", "n": 27, "block": 5, "layers": 4, "dtype": "c128"},
        # the adjoint workload: 24 qubits, 8 layers, 384 parameters
        {"name": "adjoint_24q_c128", "family": "adjoint", "n": 24, "layers": 8, "dtype": "c128"},
        # a quarter of the batch workload: n from 10 to 22, depth from 4 to 16
        {"name": "batch_64_c64", "family": "batch", "count": 64, "n_lo": 10, "n_hi": 22, "d_lo": 4, "d_hi": 16,
         "dtype": "c64"},
        # shots from a 1 GiB state
        {"name": "sample_26q_c128", "family": "sample", "n": 26, "shots": 200000, "dtype": "c128"},
        # 54 terms on a 2 GiB state
        {"name": "expect_27q_c128", "family": "expect", "n": 27, "dtype": "c128"},
        # noisy trajectories on a mid-size register
        {"name": "noisy_14q_c128", "family": "noisy", "n": 14, "layers": 3, "shots": 8, "dtype": "c128"},
    ]


def draw(rng):
    family = rng.choice(["simulate", "circuit", "circuit", "qft", "two_target", "blocks", "adjoint", "batch", "sample",
                         "expect", "noisy"])
    dtype = rng.choice(["c128", "c128", "c64"])
    if family == "simulate":
        return {"family": family, "n": rng.randint(6, 15), "layers": rng.randint(2, 10), "crz": rng.randint(0, 5),
                "shots": rng.choice([0, 10, 100, 1000]), "dtype": "c128"}
    if family == "circuit":
        n = rng.randint(14, 29)
        return {"family": family, "n": n, "layers": rng.randint(2, 10 if n > 24 else 24), "crz": rng.randint(0, n // 2),
                "dtype": dtype}
    if family == "qft":
        return {"family": family, "n": rng.randint(14, 29), "dtype": dtype}
    if family == "two_target":
        return {"family": family, "n": rng.randint(13, 27), "layers": rng.randint(2, 8), "dtype": dtype}
    if family == "blocks":
        return {"family": family, "n": rng.randint(15, 28), "block": rng.randint(4, 6), "layers": rng.randint(2, 8),
                "dtype": dtype}
    if family == "adjoint":
        return {"family": family, "n": rng.randint(8, 24), "layers": rng.randint(2, 8), "dtype": dtype}
    if family == "batch":
        lo = rng.randint(8, 16)
        return {"family": family, "count": int(round(math.exp(rng.uniform(math.log(4), math.log(64))))), "n_lo": lo,
                "n_hi": rng.randint(lo, 22), "d_lo": 4, "d_hi": rng.randint(4, 16), "dtype": dtype}
    if family == "sample":
        return {"family": family, "n": rng.randint(10, 27), "dtype": dtype,
                "shots": int(round(math.exp(rng.uniform(math.log(100), math.log(1000000)))))}
    if family == "expect":
        return {"family": family, "n": rng.randint(10, 27), "dtype": dtype}
    return {"family": family, "n": rng.randint(8, 18), "layers": rng.randint(1, 3), "shots": rng.randint(2, 12),
            "dtype": "c128"}


# --------------------------------------------------------------------------------------------- circuits
GATES = {"u3": U3Gate, "x": XGate, "h": HGate, "ry": RYGate, "rz": RZGate, "cx": CXGate, "cz": CZGate, "cp": CPGate,
         "crz": CRZGate, "swap": SwapGate, "iswap": ISwapGate, "rxx": RXXGate, "ryy": RYYGate, "cswap": CSwapGate,
         "depolarizing": Depolarizing, "damping": AmplitudeDamping}
TWO_PI = 2 * math.pi


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _brickwork(n, layers, crz, rng):
    ops = []
    for _ in range(layers):
        ang = rng.uniform(0.0, TWO_PI, size=(n, 3))
        ops += [("u3", (q,), tuple(map(float, ang[q]))) for q in range(n)]
        ops += [("cx", (2 * i, 2 * i + 1), ()) for i in range(n // 2)]
        ops += [("cx", (2 * i + 1, 2 * i + 2), ()) for i in range((n - 1) // 2)]
        for _ in range(crz):
            c, t = rng.choice(n, 2, replace=False)
            ops.append(("crz", (int(c), int(t)), (float(rng.uniform(0.0, TWO_PI)),)))
    return ops


def _qft(n, x):
    ops = [("x", (q,), ()) for q in range(n) if (x >> q) & 1]
    for j in range(n - 1, -1, -1):
        ops.append(("h", (j,), ()))
        ops += [("cp", (k, j), (TWO_PI / 2 ** (j - k + 1),)) for k in range(j - 1, -1, -1)]
    return ops


def _two_target(n, layers, rng):
    ops = []
    for _ in range(layers):
        ops += [("u3", (q,), tuple(map(float, rng.uniform(0.0, TWO_PI, 3)))) for q in range(n)]
        for k in range(n // 2):
            pair = tuple(int(v) for v in rng.choice(n, 2, replace=False))
            name = ("swap", "iswap", "rxx", "ryy")[k % 4]
            ops.append((name, pair, (float(rng.uniform(0.0, TWO_PI)),) if name in ("rxx", "ryy") else ()))
        ops.append(("cswap", tuple(int(v) for v in rng.choice(n, 3, replace=False)), ()))
    return ops


def _blocks(n, block, layers, rng):
    ops = []
    for _ in range(layers):
        ang = rng.uniform(0.0, TWO_PI, size=(n, 3))
        ops += [("u3", (q,), tuple(map(float, ang[q]))) for q in range(n)]
        for b in range(0, n, block):
            ops += [("cx", (q, q + 1), ()) for q in range(b, min(b + block, n) - 1)]
    return ops


def _ansatz(n, layers, rng):
    """RY and RZ on every qubit and a CZ ring per layer; every angle is a parameter, in gate order."""
    ops = []
    for _ in range(layers):
        ops += [("ry", (q,), (float(rng.uniform(-math.pi, math.pi)),)) for q in range(n)]
        ops += [("rz", (q,), (float(rng.uniform(-math.pi, math.pi)),)) for q in range(n)]
        ops += [("cz", (q, (q + 1) % n), ()) for q in range(n)]
    return ops


def _noisy(n, layers, rng):
    ops = []
    for _ in range(layers):
        ops += [("ry", (q,), (float(rng.uniform(-math.pi, math.pi)),)) for q in range(n)]
        ops += [("cx", (q, q + 1), ()) for q in range(n - 1)]
        ops += [("depolarizing", (q,), (0.02,)) for q in range(n)]
        ops += [("damping", (q,), (0.03,)) for q in range(n)]
    return ops


def _ops(case, seed):
    rng, family, n = _rng(seed), case["family"], case.get("n", 0)
    if family in ("simulate", "circuit"):
        return _brickwork(n, case["layers"], case["crz"], rng)
    if family == "qft":
        return _qft(n, int(rng.integers(1 << n)))
    if family == "two_target":
        return _two_target(n, case["layers"], rng)
    if family == "blocks":
        return _blocks(n, case["block"], case["layers"], rng)
    if family == "adjoint":
        return _ansatz(n, case["layers"], rng)
    return _noisy(n, case["layers"], rng)


def _batch_ops(case, seed):
    """Sizes come from the case, so that every seed has the same set of circuits with other angles."""
    shape = _rng(case["count"] * 1000 + case["n_lo"])
    rng = _rng(seed)
    out = []
    for _ in range(case["count"]):
        n = int(shape.integers(case["n_lo"], case["n_hi"] + 1))
        out.append((n, _ansatz(n, int(shape.integers(case["d_lo"], case["d_hi"] + 1)), rng)))
    return out


def _circuit(n, ops, parametrised=False, measure=False):
    qc = pq.QuantumCircuit(n)
    k = 0
    for name, qubits, angles in ops:
        if parametrised and angles:
            angles = (Parameter(f"t{k}", angles[0]),)
            k += 1
        qc << GATES[name](*qubits, *angles)
    if measure:
        qc.measure(list(range(n)))
    return qc


def _tfim(n):
    """Sum of Z_i Z_{i+1} on a ring and 0.7 X_i."""
    return [("ZZ", (i, (i + 1) % n), 1.0) for i in range(n)] + [("X", (i,), 0.7) for i in range(n)]


def _zsum(n):
    return [("Z", (i,), 1.0) for i in range(n)]


def _bloch(n):
    return [(p, (i,), 1.0) for p in "XYZ" for i in range(n)]


def _terms(case):
    n = case["n"]
    return {"qft": _bloch, "simulate": _zsum, "noisy": _zsum}.get(case["family"], _tfim)(n)


def _hamiltonian(terms):
    return Hamiltonian([PauliOp(" ".join(f"{p}{q}" for p, q in zip(s, qs)), c) for s, qs, c in terms])


def _reads_state(case):
    """Registers of at most 20 qubits (16 MiB) are read back whole."""
    return case["family"] == "circuit" and case["n"] <= 20


def _bitstrings(n, seed):
    return _rng(seed + 1).integers(1 << n, size=4096, dtype=np.uint64)


def _random_state(n, seed):
    """A Haar-like random state (what a deep random circuit leaves), complex128 on the host."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(seed)
    v = torch.randn(1 << n, 2, dtype=torch.float64, device=dev, generator=gen)
    v /= torch.linalg.vector_norm(v)
    return torch.view_as_complex(v).cpu().numpy()


# ---------------------------------------------------------------------------------------------- running
def prepare(case, seed):
    family, n, dtype = case["family"], case.get("n", 0), case["dtype"]
    if family == "batch":
        items, values = [], []
        for nq, ops in _batch_ops(case, seed):
            items.append(compile_item(_circuit(nq, ops, parametrised=True), _hamiltonian(_zsum(nq))))
            values.append(np.array([a[0] for _, _, a in ops if a]))
        return {"case": case, "runner": BatchRunner(dtype=dtype), "items": items, "values": values}
    if family in ("sample", "expect"):
        dev = _native.DeviceState(n, dtype)
        dev.load(_random_state(n, seed))
        state = {"case": case, "dev": dev}
        if family == "sample":
            state["uniforms"] = _rng(seed + 1).random(case["shots"])
        else:
            state["terms"] = [(s, list(q)) for s, q, _ in _terms(case)]
        return state
    ops = _ops(case, seed)
    if family == "adjoint":
        values = [a[0] for _, _, a in ops if a]
        return {"case": case, "qc": _circuit(n, ops, parametrised=True), "hamiltonian": _hamiltonian(_terms(case)),
                "params": torch.tensor(values, dtype=torch.float64, requires_grad=True)}
    if family in ("simulate", "noisy"):
        return {"case": case, "qc": _circuit(n, ops, measure=True), "hamiltonian": _hamiltonian(_terms(case)),
                "seed": seed}
    return {"case": case, "dev": _native.DeviceState(n, dtype), "prog": compile_circuit(_circuit(n, ops)),
            "terms": [(s, list(q)) for s, q, _ in _terms(case)], "bitstrings": _bitstrings(n, seed)}


def run(state):
    case = state["case"]
    family = case["family"]
    if family in ("simulate", "noisy"):
        kind = "statevector" if family == "simulate" else "noisy statevetor"
        res = simulate(state["qc"], simulator=kind, shots=case["shots"], hamiltonian=state["hamiltonian"],
                       precision=case["dtype"], seed=state["seed"])
        counts = np.zeros(1 << case["n"], dtype=np.int64)
        for key, times in res["counts"].items():
            counts[int(key, 2)] = times
        out = {"expects": np.array(res["pauli_expects"], dtype=np.float64), "counts": counts}
        if family == "simulate":
            out["state"] = res.get_statevector()
        return out
    if family == "adjoint":
        loss = expectation(state["qc"], state["hamiltonian"], state["params"], precision=case["dtype"])
        (grads,) = torch.autograd.grad(loss, state["params"])
        return {"loss": loss.detach(), "grads": grads}
    if family == "batch":
        results, _ = state["runner"].run(state["items"], state["values"])
        return {"losses": np.array([r.expectation for r in results]), "grads": np.concatenate([r.grads for r in results])}
    dev = state["dev"]
    if family == "sample":
        return dev.sample(state["uniforms"])
    if family == "expect":
        return dev.expect(state["terms"])
    dev.init_zero()
    dev.apply(state["prog"])
    if _reads_state(case):
        return dev.store()
    return {"amplitudes": dev.gather(state["bitstrings"]), "expects": dev.expect(state["terms"])}


# ------------------------------------------------------------------------------------------------- work
FLOPS = {"u3": 14, "x": 0, "h": 6, "ry": 6, "rz": 6, "cx": 0, "cz": 0.5, "cp": 1.5, "crz": 3, "swap": 0, "iswap": 0.5,
         "rxx": 6, "ryy": 6, "cswap": 0, "depolarizing": 0, "damping": 3}  # per amplitude of the register


def _gate_flops(n, ops):
    return sum(FLOPS[name] for name, _, _ in ops) * 2.0 ** n


def work(case):
    family, n = case["family"], case.get("n", 0)
    amp = 16 if case["dtype"] == "c128" else 8
    if family == "batch":
        by = fl = 0.0
        for nq, ops in _batch_ops(case, 0):  # psi and lambda, each written once and read once
            by += 4.0 * amp * 2.0 ** nq
            fl += 3 * _gate_flops(nq, ops)
        return {"bytes": by, "flops": fl}
    size = amp * 2.0 ** n
    if family == "sample":
        return {"bytes": size + case["shots"] * 16.0, "flops": 4.0 * 2.0 ** n}
    if family == "expect":
        return {"bytes": size, "flops": (4.0 + 2.0 * len(_terms(case))) * 2.0 ** n}
    ops = _ops(case, 0)
    if family == "adjoint":
        return {"bytes": 4 * size, "flops": 3 * _gate_flops(n, ops)}
    by, fl = 2 * size, _gate_flops(n, ops) + 2.0 * len(_terms(case)) * 2.0 ** n
    if family == "noisy":
        by, fl = by * case["shots"], fl * case["shots"]
    return {"bytes": by, "flops": fl}


# ------------------------------------------------------------------------------------------------ exact
# Plain 64-bit evaluation with torch (on the GPU where there is one; without one only small registers
# are worth the time).

EXACT_MAX = 27


def _u3(theta, phi, lam):
    c, s = math.cos(theta / 2), math.sin(theta / 2)
    return np.array([[c, -np.exp(1j * lam) * s], [np.exp(1j * phi) * s, np.exp(1j * (phi + lam)) * c]])


def _matrix(name, angles):
    """(number of controls, matrix whose index bit j belongs to target j)."""
    if name == "u3":
        return 0, _u3(*angles)
    if name in ("x", "cx"):
        return int(name == "cx"), np.array([[0, 1], [1, 0]], dtype=complex)
    if name == "h":
        return 0, np.array([[1, 1], [1, -1]], dtype=complex) / math.sqrt(2)
    if name == "ry":
        c, s = math.cos(angles[0] / 2), math.sin(angles[0] / 2)
        return 0, np.array([[c, -s], [s, c]], dtype=complex)
    if name in ("rz", "crz"):
        return int(name == "crz"), np.diag(np.exp([-0.5j * angles[0], 0.5j * angles[0]]))
    if name == "cz":
        return 1, np.diag([1.0 + 0j, -1.0])
    if name == "cp":
        return 1, np.diag([1.0 + 0j, np.exp(1j * angles[0])])
    if name in ("swap", "cswap", "iswap"):
        m = np.eye(4, dtype=complex)
        e = 1j if name == "iswap" else 1.0
        m[1:3, 1:3] = [[0, e], [e, 0]]
        return int(name == "cswap"), m
    c, s = math.cos(angles[0] / 2), 1j * math.sin(angles[0] / 2)
    m = np.diag([c + 0j] * 4)
    m[0, 3] = m[3, 0] = -s if name == "rxx" else s
    m[1, 2] = m[2, 1] = -s
    return 0, m


def _slices(psi, n, qubits):
    """psi as a view with one axis of length 2 per named qubit, and those axes' positions."""
    shape, axis, top = [], {}, n
    for q in sorted(qubits, reverse=True):
        shape.append(1 << (top - 1 - q))
        axis[q] = len(shape)
        shape.append(2)
        top = q
    shape.append(1 << top)
    return psi.view(shape), axis


def _apply_matrix(psi, n, ctrls, targets, m):
    view, axis = _slices(psi, n, list(ctrls) + list(targets))
    parts = []
    for r in range(len(m)):
        idx = [slice(None)] * view.dim()
        for c in ctrls:
            idx[axis[c]] = 1
        for j, t in enumerate(targets):
            idx[axis[t]] = (r >> j) & 1
        parts.append(tuple(idx))
    old = [view[p].clone() for p in parts]
    for r, p in enumerate(parts):
        if m[r, r] == 1 and np.count_nonzero(m[r]) == 1:
            continue  # this slice keeps its values
        acc = torch.zeros_like(old[r])
        for c in np.flatnonzero(m[r]):
            acc += old[c] * complex(m[r, c])
        view[p] = acc


def _apply(psi, n, op, dagger=False):
    name, qubits, angles = op
    nc, m = _matrix(name, angles)
    _apply_matrix(psi, n, qubits[:nc], qubits[nc:], m.conj().T if dagger else m)


PAULI = {"X": np.array([[0, 1], [1, 0]], dtype=complex), "Y": np.array([[0, -1j], [1j, 0]]),
         "Z": np.diag([1.0 + 0j, -1.0])}


def _pauli(psi, n, letters, qubits):
    out = psi.clone()
    for p, q in zip(letters, qubits):
        _apply_matrix(out, n, (), (q,), PAULI[p])
    return out


def _dot(a, b):
    """<a|b>."""
    return complex(torch.vdot(a, b))


def _expects(psi, n, terms):
    return np.array([_dot(psi, _pauli(psi, n, s, q)).real for s, q, _ in terms])


def _zero_state(n, device):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=device)
    psi[0] = 1.0
    return psi


def _adjoint(n, ops, terms, device):
    psi = _zero_state(n, device)
    for op in ops:
        _apply(psi, n, op)
    lam = torch.zeros_like(psi)
    for s, q, c in terms:
        lam += c * _pauli(psi, n, s, q)
    loss = _dot(psi, lam).real
    grads = []
    for op in reversed(ops):
        if op[2]:
            grads.append(_dot(lam, _pauli(psi, n, op[0][1].upper(), op[1])).imag)
        _apply(psi, n, op, dagger=True)
        _apply(lam, n, op, dagger=True)
    return loss, np.array(grads[::-1])


def _qft_amplitudes(n, x, y):
    """2^(-n/2) e^{2 pi i x rev(y) / 2^n}, the phase as an integer mod 2^n."""
    rev = np.zeros_like(y)
    for b in range(n):
        rev |= ((y >> np.uint64(b)) & np.uint64(1)) << np.uint64(n - 1 - b)
    phase = (np.uint64(x) * rev) & np.uint64((1 << n) - 1)  # products wrap mod 2^64, a multiple of 2^n
    return np.exp(2j * np.pi * (phase.astype(np.float64) / (1 << n))) / math.sqrt(1 << n)


def _qft_bloch(n, x):
    """The QFT of a basis state is a product state: qubit j is (|0> + e^{2 pi i x / 2^(j + 1)} |1>) / sqrt 2."""
    phase = [TWO_PI * (x % (1 << (j + 1))) / (1 << (j + 1)) for j in range(n)]
    return np.array([math.cos(p) for p in phase] + [math.sin(p) for p in phase] + [0.0] * n)


def _trajectories(case, seed, device):
    """The noisy run's rule: per shot one uniform per channel in circuit order, then one for the
    sample. Depolarizing picks X, Y, Z or nothing by cumulative probability; damping takes operator k
    with the first running sum of |K_j psi| / |psi| above the uniform."""
    n, ops, terms = case["n"], _ops(case, seed), _terms(case)
    rng = np.random.default_rng(seed)
    channels = sum(name in ("depolarizing", "damping") for name, _, _ in ops)
    total = np.zeros(len(terms))
    for _ in range(case["shots"]):
        u = iter(rng.random(channels + 1))
        psi = _zero_state(n, device)
        for op in ops:
            name, (q, *_), angles = op
            if name == "depolarizing":
                p, x = angles[0], next(u)
                for k, letter in enumerate("XYZ"):
                    if x < (k + 1) * p / 3:
                        _apply_matrix(psi, n, (), (q,), PAULI[letter])
                        break
            elif name == "damping":
                p, x, acc = angles[0], next(u), 0.0
                norm = float(torch.linalg.vector_norm(psi))
                for m in (np.diag([1.0 + 0j, math.sqrt(1 - p)]), np.array([[0, math.sqrt(p)], [0, 0]], dtype=complex)):
                    trial = psi.clone()
                    _apply_matrix(trial, n, (), (q,), m)
                    size = float(torch.linalg.vector_norm(trial))
                    acc += size / norm
                    if x < acc:
                        psi = trial / size
                        break
            else:
                _apply(psi, n, op)
        next(u)
        total += _expects(psi, n, terms)
    return total / case["shots"]


def exact(case, seed):
    family, n = case["family"], case.get("n", 0)
    gpu = torch.cuda.is_available()
    device = "cuda" if gpu else "cpu"
    if family == "sample":
        return None  # indices: whole numbers
    if family == "qft":
        x = int(_rng(seed).integers(1 << n))
        return {"amplitudes": _qft_amplitudes(n, x, _bitstrings(n, seed)), "expects": _qft_bloch(n, x)}
    if family == "batch":
        if not gpu:
            return None
        done = [_adjoint(nq, ops, _zsum(nq), device) for nq, ops in _batch_ops(case, seed)]
        return {"losses": np.array([e for e, _ in done]), "grads": np.concatenate([g for _, g in done])}
    if n > (EXACT_MAX if gpu else 16) and family != "expect":
        return None
    if family == "expect":
        if n > 20 and not gpu:
            return None
        psi = torch.from_numpy(_random_state(n, seed)).to(device)
        return _expects(psi, n, _terms(case))
    if family == "adjoint":
        loss, grads = _adjoint(n, _ops(case, seed), _terms(case), device)
        return {"loss": torch.tensor(loss, dtype=torch.float64), "grads": torch.from_numpy(grads)}
    if family == "noisy":
        return {"expects": _trajectories(case, seed, device), "counts": None}
    psi = _zero_state(n, device)
    for op in _ops(case, seed):
        _apply(psi, n, op)
    if family == "simulate":
        return {"expects": _expects(psi, n, _terms(case)), "counts": None, "state": psi.cpu().numpy()}
    if _reads_state(case):
        return psi.cpu().numpy()
    at = torch.from_numpy(_bitstrings(n, seed).astype(np.int64)).to(device)
    return {"amplitudes": psi[at].cpu().numpy(), "expects": _expects(psi, n, _terms(case))}
