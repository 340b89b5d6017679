"""Plans whose tiles have one chosen qubit beside the low ones (low_bits = tile_bits - 1): dense gates on two
high qubits, which such a tile cannot hold, and layouts, which it could not restore. On the CPU, replayed
against the oracle; a pass that takes no gate is an error, so a plan always ends."""

import numpy as np
import pytest

from oracle.cpu import CpuState
from pyquafu_amd import _native
from pyquafu_amd.simulators.program import GENERAL, MULTI, ProgramBuilder
from tests.conftest import rand_state
from tests.progs import random_unitary
from tests.test_planner import replay


def _check(prog, n, dtype="c128", **kw):
    plan = _native.plan_json(prog, n, dtype, **kw)
    assert all(it["groups"] or it["out_bit"] for it in plan["items"] if it["fused"])
    psi0 = rand_state(n, np.random.Generator(np.random.PCG64(n)))
    cpu = CpuState(n)
    cpu.load(psi0)
    cpu.apply(prog)
    # (collapsed: items outside passes are dense gates with the matrix that the plan gives)
    assert np.abs(replay(plan, prog, n, psi0, collapsed=True) - cpu.store()).max() < 1e-12


@pytest.mark.parametrize("layout", [False, True])
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("extra", [1, 2, 4])
@pytest.mark.parametrize("tile", [9, 10, 11, 12, 13])
def test_two_target_gates_on_high_qubits(tile, extra, dtype, layout):
    n = tile + extra
    rng = np.random.Generator(np.random.PCG64(100 * n + tile))
    b = ProgramBuilder()
    for k in range(12):
        pair = [n - 1, tile - 1] if k % 3 == 0 else [int(x) for x in rng.choice(n, 2, replace=False)]
        b.add(MULTI, pair, matrix=random_unitary(4, rng))
        b.add(GENERAL, [int(rng.integers(n))], matrix=random_unitary(2, rng))
    _check(b.program(n_qubits=n), n, dtype, tile_bits=tile, low_bits=tile - 1, layout=layout)


# (one free qubit: the plans of these seeds end with two or more high qubits in each other's places)
@pytest.mark.parametrize("free,seed", [(1, 15), (1, 32), (1, 39), (1, 49), (1, 56), (2, 15), (2, 32), (3, 39)])
def test_layout_of_few_free_qubits_is_restored(free, seed):
    rng = np.random.Generator(np.random.PCG64(40 * seed + 1))
    tile = int(rng.integers(9, 12))
    n = tile + int(rng.integers(3, 7))
    b = ProgramBuilder()
    for _ in range(int(rng.integers(20, 60))):
        nc = int(rng.choice([0, 0, 1, 1, 2]))
        q = [int(x) for x in rng.choice(n, nc + 1, replace=False)]
        b.add(GENERAL, q, n_ctrl=nc, matrix=random_unitary(2, rng))
    _check(b.program(n_qubits=n), n, tile_bits=tile, low_bits=tile - free, layout=True)
