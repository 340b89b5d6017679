"""Runs of Kraus channels with diagonal K^H K on different qubits, which are decided from one set of joint
populations, against the dense oracle with the same uniforms."""

from contextlib import closing

import numpy as np
import pytest

import pyquafu_amd as pq
from oracle import dense
from pyquafu_amd import _native
from pyquafu_amd.elements import AmplitudeDamping, BitFlip, Decoherence, Depolarizing, KrausChannel, QuantumGate
from pyquafu_amd.simulators.simulator import NoiseSVSimulator
from tests.conftest import rand_state
from tests.test_gpu_noise import TOL, random_kraus

pytestmark = pytest.mark.gpu


def _runs(n, rng):
    """Damping on every qubit (a run, two from 15 qubits), then mixes: unitary channels within a run, on a
    qubit of it and before a later one, a qubit named twice, a set that leaves no branch, gates and
    general Kraus sets between."""
    qc = pq.QuantumCircuit(n)
    for q in range(n):
        qc.ry(q, float(rng.uniform(-3, 3)))
    for q in rng.permutation(n):
        qc << AmplitudeDamping(int(q), float(rng.uniform(0.2, 0.9)))  # noqa
    for step in range(3 * min(n, 8)):
        q = int(rng.integers(n))
        kind = step % 6
        if kind in (0, 3):
            qc << AmplitudeDamping(q, float(rng.uniform(0.2, 0.9)))  # noqa
        elif kind == 1:
            qc << [BitFlip, Depolarizing][int(rng.integers(2))](q, 0.5)  # noqa
        elif kind == 2:
            qc << Decoherence(q, 1.5, 3.0, 2.5)  # noqa
        elif kind == 4:
            qc << [KrausChannel("h", q, [QuantumGate("H", [q], [], 0.5 * np.eye(2, dtype=complex))]),
                   random_kraus(q, 2, rng)][int(rng.integers(2))]  # noqa
        else:
            qc.rx(q, float(rng.uniform(-3, 3)))
    return qc


# 8 qubits are the thread index; 9 to 16 leave qubits above it, 16 exceeds one run
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 14, 16])
def test_kraus_runs(n, dtype):
    rng = np.random.Generator(np.random.PCG64(8200 + n))
    prog = NoiseSVSimulator.trajectory_program(_runs(n, rng))
    with closing(_native.DeviceState(n, dtype)) as dev:
        for _ in range(3):
            u = rng.random(prog.n_random)
            psi0 = rand_state(n, rng)
            dev.load(psi0)
            dev.run(prog, u, 0, True)
            want, _ = dense.run_dense(prog, n, psi=psi0, uniforms=u)
            assert np.abs(dev.store() - want).max() < TOL[dtype] * 10


# asked qubits below, above and on both sides of the thread index; slices to sum but in the last two
@pytest.mark.parametrize("qubits", [[0], [9], [19], [0, 1, 2, 3, 4, 5, 6, 7], [3, 7, 8, 11, 19], list(range(6, 20))])
def test_kraus_run_on_some_qubits(qubits):
    n = 20
    rng = np.random.Generator(np.random.PCG64(8300 + sum(qubits)))
    qc = pq.QuantumCircuit(n)
    for q in qubits:
        qc << AmplitudeDamping(q, 0.8)  # noqa
    prog = NoiseSVSimulator.trajectory_program(qc)
    u = rng.random(prog.n_random)
    psi0 = rand_state(n, rng)
    with closing(_native.DeviceState(n, "c128")) as dev:
        dev.load(psi0)
        dev.run(prog, u, 0, True)
        want, _ = dense.run_dense(prog, n, psi=psi0, uniforms=u)
        assert np.abs(dev.store() - want).max() < 1e-11
