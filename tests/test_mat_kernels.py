"""Matrix-core passes themselves: lists whose plans are made of them (asserted), with gates that widen groups by
their controls, matrices that differ within a wavefront, single gates between the passes and 4x4 ops with
outside controls. On the CPU the plans are replayed against the oracle, on the GPU the states are compared.

Tolerance: the engine's complex128 bound, 1e-12 max-abs on unit-norm states (see test_mat_passes)."""

import numpy as np
import pytest

from oracle.cpu import CpuState
from pyquafu_amd import _native
from pyquafu_amd.simulators.program import CCX, GENERAL, MULTI, ProgramBuilder
from tests.conftest import rand_state
from tests.progs import random_unitary
from tests.test_planner import replay

TOL = 1e-12
G_MULTI, G_SWAP, G_DIAG = 4, 3, 2


def program(n, rng, count, most, wide=0):
    """`count` gates with up to `most` controls, half of them dense; every `wide`-th gate has 7."""
    b = ProgramBuilder()
    for k in range(count):
        nc = 7 if wide and k % wide == wide - 1 else int(rng.integers(0, most + 1))
        kind = rng.random()
        nt = 2 if kind < 0.2 else 1
        q = [int(x) for x in rng.choice(n, nc + nt, replace=False)]
        if nt == 2:
            b.add(MULTI, q, n_ctrl=nc, matrix=random_unitary(4, rng))
        elif kind < 0.6:
            b.add(GENERAL, q, n_ctrl=nc, matrix=random_unitary(2, rng))
        elif kind < 0.8:
            b.add(GENERAL, q, n_ctrl=nc, matrix=np.diag(np.exp(1j * rng.uniform(-3, 3, 2))))
        elif nc == 2:
            b.add(CCX, q)
        else:
            b.add(GENERAL, q, n_ctrl=nc, matrix=np.array([[0, 1], [1, 0]], dtype=complex))
    return b.program(n_qubits=n)


def as_dense(plan):
    """Items outside passes as dense gates with their matrix, as replay takes them."""
    for it in plan["items"]:
        if not it["fused"] and it["kind"] != G_MULTI:
            m = [[0, 0], [1, 0], [1, 0], [0, 0]] if it["kind"] == G_SWAP else it["m"]
            if it["kind"] == G_DIAG:
                m = [it["m"][0], [0, 0], [0, 0], it["m"][1]]
            it.update(kind=G_MULTI, targets=[it["target"]], m=m)
    return plan


# n, tile, low, controls: tiles of 9 to 13 bits, whole states, one and two free qubits, several tiles
SHAPES = [(9, 0, 0, 1), (10, 9, 3, 1), (10, 9, 8, 1), (11, 9, 7, 1), (11, 10, 9, 1), (12, 0, 0, 3), (13, 0, 0, 3),
          (13, 11, 10, 2), (14, 13, 3, 3), (15, 10, 4, 2), (15, 13, 12, 2), (16, 12, 5, 3), (17, 11, 3, 2)]


def make(n, tile, low, controls, wide=0):
    rng = np.random.Generator(np.random.PCG64(31 * n + tile + low))
    prog = program(n, rng, 6 * n, controls, wide)
    return prog, rand_state(n, rng)


def oracle(prog, n, psi0):
    cpu = CpuState(n)
    cpu.load(psi0)
    cpu.apply(prog)
    return cpu.store()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,tile,low,controls", SHAPES)
def test_plan_replays(n, tile, low, controls, layout):
    prog, psi0 = make(n, tile, low, controls)
    plan = as_dense(_native.plan_json(prog, n, tile_bits=tile, low_bits=low, layout=layout))
    assert all(it["mat"] for it in plan["items"] if it["fused"])
    assert np.abs(replay(plan, prog, n, psi0, collapsed=True) - oracle(prog, n, psi0)).max() < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,tile,low,controls", SHAPES)
def test_kernel_matches_oracle(n, tile, low, controls, layout):
    prog, psi0 = make(n, tile, low, controls)
    dev = _native.DeviceState(n, "c128")
    for key, value in (("tile_bits", tile), ("low_bits", low), ("layout", layout), ("dense_blocks", 0)):
        dev.set_option(key, value)
    dev.load(psi0)
    dev.apply(prog)
    got, prof = dev.store(), dev.profile()
    dev.close()
    assert "mat_build" in prof
    assert np.abs(got - oracle(prog, n, psi0)).max() < TOL


# a few gates with seven controls, which no group holds, between the passes (32 and 64 tiles)
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,wide", [(17, 50), (18, 50)])
def test_single_gates_between_passes(n, wide, layout):
    prog, psi0 = make(n, 0, 0, 1, wide)
    plan = as_dense(_native.plan_json(prog, n, layout=layout))
    items = plan["items"]
    assert all(it["mat"] for it in items if it["fused"]) and not all(it["fused"] for it in items)
    assert np.abs(replay(plan, prog, n, psi0, collapsed=True) - oracle(prog, n, psi0)).max() < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,wide", [(17, 50), (18, 50)])
def test_single_gates_between_kernels(n, wide, layout):
    prog, psi0 = make(n, 0, 0, 1, wide)
    dev = _native.DeviceState(n, "c128")
    dev.set_option("layout", layout)
    dev.set_option("dense_blocks", 0)
    dev.load(psi0)
    dev.apply(prog)
    got, prof = dev.store(), dev.profile()
    dev.close()
    assert "mat_build" in prof and prof.keys() - {"mat_build", "fused_pass"}
    assert np.abs(got - oracle(prog, n, psi0)).max() < TOL


@pytest.mark.gpu
def test_plan_of_several_segments():
    """More matrices than are built at a time (2^15): two uploads and two launches of the builder in one call."""
    n = 13
    rng = np.random.Generator(np.random.PCG64(77))
    prog = program(n, rng, 16000, 3)
    psi0 = rand_state(n, rng)
    dev = _native.DeviceState(n, "c128")
    dev.load(psi0)
    dev.apply(prog)
    got, prof = dev.store(), dev.profile()
    dev.close()
    assert prof["mat_build"]["launches"] >= 2
    # 16,000 gates: each rounds its two products to some 2^-53 of amplitudes of norm 1 in all
    assert np.abs(got - oracle(prog, n, psi0)).max() < 1e-11
