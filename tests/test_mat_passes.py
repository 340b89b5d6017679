"""Matrix-core passes (complex128 one-state passes whose groups are 8x8 matrices): the plans on the CPU,
replayed against the oracle, and the kernels on the GPU, against the oracle and the vector kernels.

The tolerance is the engine's complex128 bound (1e-12 max-abs on unit-norm states): a matrix of a
group is a product of at most a few hundred gates in double precision (relative error below 1e-13)
and a row's product adds 16 terms of magnitude at most 1."""

import numpy as np
import pytest

from oracle.cpu import CpuState
from pyquafu_amd import _native, workloads
from pyquafu_amd.simulators.program import CCX, GENERAL, MULTI, ProgramBuilder, compile_circuit
from tests.conftest import rand_state
from tests.progs import random_gate_program, random_unitary
from tests.test_planner import check

TOL = 1e-12


def wide_program(n, rng, most):
    """Gates with 0 .. most controls (dense, diagonal, X, dense on two targets) between layers that
    spread over the register: more outside qubits than a group may have, groups that have to take
    controls in, gates that no group holds."""
    b = ProgramBuilder()
    for _ in range(60):
        nc = int(rng.integers(0, most + 1))
        nt = 2 if rng.random() < 0.25 else 1
        q = [int(x) for x in rng.choice(n, nc + nt, replace=False)]
        kind = rng.random()
        if nt == 2:
            b.add(MULTI, q, n_ctrl=nc, matrix=random_unitary(4, rng))
        elif kind < 0.4:
            b.add(GENERAL, q, n_ctrl=nc, matrix=random_unitary(2, rng))
        elif kind < 0.7:
            b.add(GENERAL, q, n_ctrl=nc, matrix=np.diag(np.exp(1j * rng.uniform(-3, 3, 2))))
        elif nc == 2:
            b.add(CCX, q)
        else:
            b.add(GENERAL, q, n_ctrl=nc, matrix=np.array([[0, 1], [1, 0]], dtype=complex))
    return b.program(n_qubits=n)


SHAPES = [(9, 0, 0), (10, 9, 3), (11, 9, 8), (12, 0, 0), (13, 0, 0), (14, 13, 3), (15, 10, 4), (16, 12, 5)]


@pytest.mark.parametrize("layout", [False, True])
@pytest.mark.parametrize("n,tile,low", SHAPES)
def test_wide_gates_plan_replays(n, tile, low, layout):
    prog = wide_program(n, np.random.Generator(np.random.PCG64(n + tile)), min(7, n - 2))
    check(prog, n, tile_bits=tile, low_bits=low, layout=layout)


def run_gpu(prog, n, psi0, **options):
    dev = _native.DeviceState(n, "c128")
    for key, value in options.items():
        dev.set_option(key, value)
    dev.load(psi0)
    dev.apply(prog)
    got, prof = dev.store(), dev.profile()
    dev.close()
    return got, prof


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,tile,low", SHAPES)
def test_wide_gates_match_oracle(n, tile, low, layout):
    rng = np.random.Generator(np.random.PCG64(n + tile))
    for prog in (wide_program(n, rng, min(7, n - 2)), random_gate_program(n, 200, rng, max_multi=3)):
        psi0 = rand_state(n, rng)
        cpu = CpuState(n)
        cpu.load(psi0)
        cpu.apply(prog)
        want = cpu.store()
        got, prof = run_gpu(prog, n, psi0, tile_bits=tile, low_bits=low, layout=layout)
        assert np.abs(got - want).max() < TOL
        vec, vprof = run_gpu(prog, n, psi0, tile_bits=tile, low_bits=low, layout=layout, mfma=0)
        assert np.abs(vec - want).max() < TOL
        assert "mat_build" not in vprof


@pytest.mark.gpu
def test_mostly_diagonal_lists_keep_the_vector_kernels():
    """A QFT takes the vector passes, a brickwork the matrix-core passes, both from one handle's cache."""
    n = 18
    dev = _native.DeviceState(n, "c128")
    for prog, mat in ((compile_circuit(workloads.qft(n, 12345)), False),
                      (compile_circuit(workloads.random_u3_cx(n, 3, 4, seed=5, measure=False)), True)) * 2:
        dev.init_zero()
        dev.apply(prog)
        cpu = CpuState(n)
        cpu.apply(prog)
        assert np.abs(dev.store() - cpu.store()).max() < TOL
        assert ("mat_build" in dev.profile(reset=True)) == mat
    dev.close()
