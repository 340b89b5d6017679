"""Which gate lists run on the matrix cores: the plans' kind of passes on the CPU (qfvm_plan_json). The sides
that a list belongs to are those that were faster when timed, by a quarter or more."""

import numpy as np
import pytest

from pyquafu_amd import _native, workloads
from pyquafu_amd.simulators.program import CX, GENERAL, H, ProgramBuilder, compile_circuit
from tests.progs import random_unitary


def _mat(prog, n):
    fused = [it["mat"] for it in _native.plan_json(prog, n)["items"] if it["fused"]]
    assert len(set(fused)) == 1
    return fused[0]


def _cx(n, count):
    rng = np.random.Generator(np.random.PCG64(n * 100 + count))
    b = ProgramBuilder()
    for _ in range(count):
        b.add(CX, [int(x) for x in rng.choice(n, 2, replace=False)], n_ctrl=1)
    return b.program(n_qubits=n)


@pytest.mark.parametrize("n,count", [(11, 8), (13, 8), (14, 8), (22, 8), (22, 16), (28, 16)])
def test_short_cx_lists_keep_the_vector_kernels(n, count):
    assert not _mat(_cx(n, count), n)


@pytest.mark.parametrize("n", [18, 24, 28])
def test_qft_keeps_the_vector_kernels(n):
    assert not _mat(compile_circuit(workloads.qft(n, 12345)), n)


@pytest.mark.parametrize("n,layers", [(12, 3), (20, 2), (28, 4)])
def test_brickworks_take_the_matrix_cores(n, layers):
    assert _mat(compile_circuit(workloads.random_u3_cx(n, layers, 4, seed=5, measure=False)), n)


@pytest.mark.parametrize("n", [16, 20, 26])
def test_a_layer_that_saves_a_pass_takes_the_matrix_cores(n):
    b = ProgramBuilder()
    rng = np.random.Generator(np.random.PCG64(n))
    for q in range(12):
        b.add(GENERAL, [q], matrix=random_unitary(2, rng)) if q % 2 else b.add(H, [q])
    assert _mat(b.program(n_qubits=n), n)


@pytest.mark.parametrize("n", [14, 20])
def test_layout_option_defaults(n):
    """-1, the default of option "layout": on where the list runs on the matrix cores, off elsewhere."""
    brick = compile_circuit(workloads.random_u3_cx(n, 6, 4, seed=5, measure=False))
    plans = [_native.plan_json(brick, n, layout=v) for v in (-1, 1, 0)]
    assert plans[0] == plans[1] != plans[2]
    qft = compile_circuit(workloads.qft(20, 12345))
    plans = [_native.plan_json(qft, 20, layout=v) for v in (-1, 0, 1)]
    assert plans[0] == plans[1] != plans[2]


@pytest.mark.gpu
def test_layout_option_set_back():
    n = 20
    prog = compile_circuit(workloads.random_u3_cx(n, 6, 4, seed=5, measure=False))
    dev = _native.DeviceState(n, "c128")
    passes = []
    for value in (None, 0, 1, -1):
        if value is not None:
            dev.set_option("layout", value)
        dev.profile(reset=True)
        dev.apply(prog)
        passes.append(dev.profile(reset=True)["fused_pass"]["launches"])
    dev.close()
    assert passes[0] == passes[2] == passes[3] != passes[1]
