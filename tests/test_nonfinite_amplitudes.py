"""Infinities and NaN in the state under matrix-core passes: gates that only move or scale amplitudes carry them
along, gates that mix two amplitudes spread them to those two, and nothing else changes."""

import numpy as np
import pytest

from pyquafu_amd import _native
from pyquafu_amd.simulators.program import CP, CX, CZ, GENERAL, RZ, H, S, X, ProgramBuilder
from tests.conftest import rand_state

pytestmark = pytest.mark.gpu


def _program(n, mixing, rng):
    """A list of gates and what each does to a set of marked amplitudes (a boolean array over the indices)."""
    b = ProgramBuilder()
    steps = []
    idx = np.arange(1 << n)
    for q in range(6):  # enough non-diagonal, non-X gates for a matrix-core plan: products of 1 and phases
        b.add(GENERAL, [q], matrix=np.array([[0, 1j], [1, 0]]))
        steps.append(lambda marked, q=q: marked[idx ^ (1 << q)])
    for _ in range(5 * n):
        kind = int(rng.integers(5))
        q = [int(x) for x in rng.choice(n, 2, replace=False)]
        if kind == 0:
            b.add(X, q[:1])
            steps.append(lambda marked, t=q[0]: marked[idx ^ (1 << t)])
        elif kind == 1:
            b.add(CX, q, n_ctrl=1)
            steps.append(lambda marked, c=q[0], t=q[1]: marked[np.where((idx >> c) & 1, idx ^ (1 << t), idx)])
        elif kind == 2:
            b.add(GENERAL, q[:1], matrix=np.array([[0, 1j], [1, 0]]))
            steps.append(lambda marked, t=q[0]: marked[idx ^ (1 << t)])
        else:
            code, ctrl = [(CZ, 1), (CP, 1), (RZ, 0), (S, 0)][int(rng.integers(4))]
            b.add(code, q if ctrl else q[:1], n_ctrl=ctrl, param=0.3)
    if mixing:
        b.add(H, [mixing])
        steps.append(lambda marked, t=mixing: marked | marked[idx ^ (1 << t)])
    return b.program(n_qubits=n), steps


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, complex(0, np.inf), complex(np.nan, 1)])
@pytest.mark.parametrize("mixing", [0, 4])
@pytest.mark.parametrize("n", [9, 12, 14])
def test_nonfinite_amplitudes_stay_in_place(n, mixing, value):
    rng = np.random.Generator(np.random.PCG64(500 + n))
    prog, steps = _program(n, mixing, rng)
    psi = rand_state(n, rng)
    marked = np.zeros(1 << n, bool)
    marked[rng.choice(1 << n, 3, replace=False)] = True
    dev = _native.DeviceState(n, "c128")
    dev.load(psi)
    dev.apply(prog)
    clean = dev.store()
    bad = psi.copy()
    bad[marked] = value
    dev.load(bad)
    dev.profile(reset=True)
    dev.apply(prog)
    got = dev.store()
    assert "mat_build" in dev.profile()
    dev.close()
    for step in steps:
        marked = step(marked)
    assert np.array_equal(~np.isfinite(got), marked)
    # the others do not depend on the marked ones: as in the run without them, to rounding (entries of a
    # group's matrix are products of at most 5 n unit phases; a result adds up at most 16 terms)
    assert np.abs(got - clean)[~marked].max() < 1e-13


# states of 2^24 amplitudes and more take a kernel instance of their own
def test_nonfinite_amplitudes_of_large_states():
    n = 24
    rng = np.random.Generator(np.random.PCG64(24))
    b = ProgramBuilder()
    at = rng.choice(1 << n, 5, replace=False)
    marked = at.copy()
    for k in range(5 * n):
        q = [int(x) for x in rng.choice(n, 2, replace=False)]
        if k % 3 == 0:
            b.add(GENERAL, q[:1], matrix=np.array([[0, 1j], [1, 0]]))
            marked ^= 1 << q[0]
        elif k % 3 == 1:
            b.add(CX, q, n_ctrl=1)
            marked ^= ((marked >> q[0]) & 1) << q[1]
        else:
            b.add(CP, q, n_ctrl=1, param=0.3)
    prog = b.program(n_qubits=n)
    psi = np.full(1 << n, 2.0 ** (-n / 2), complex)
    dev = _native.DeviceState(n, "c128")
    dev.load(psi)
    dev.apply(prog)
    clean = dev.store()
    psi[at] = [np.inf, -np.inf, np.nan, complex(0, np.inf), np.inf]
    dev.load(psi)
    dev.profile(reset=True)
    dev.apply(prog)
    got = dev.store()
    assert "mat_build" in dev.profile()
    dev.close()
    bad = ~np.isfinite(got)
    assert np.array_equal(np.flatnonzero(bad), np.sort(marked))
    assert np.abs(got - clean)[~bad].max() < 1e-13
