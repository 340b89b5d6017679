"""Gradient stages of the two-state sweep that hold markers on every qubit: X, Y and Z on every tile bit, Z
outside the tile, and controlled ones between them, against the oracle."""

import numpy as np
import pytest

from oracle import gradients as og
from pyquafu_amd.simulators.program import CZ, GENERAL, RX, RY, RZ, ProgramBuilder
from tests.progs import _rot, random_pauli_terms
from tests.test_gpu_gradients import engine_adjoint

pytestmark = pytest.mark.gpu


# two-state tiles hold 2^(tile - 1) amplitudes; 10 to 12 bits are the split-row kernel's, where the top
# three bits overlap the third group (10, 11) or follow it (12). complex64 states carry 24 bits: the gradients'
# tolerance there is the other complex64 gradient tests'
@pytest.mark.parametrize("dtype,tol", [("c128", 1e-10), ("c64", 1e-4)])
@pytest.mark.parametrize("n,tile,low", [(10, 0, 0), (11, 11, 3), (12, 12, 3), (13, 13, 3), (14, 0, 0), (15, 13, 6)])
def test_full_stages(n, tile, low, dtype, tol):
    rng = np.random.Generator(np.random.PCG64(1700 + n + tile))
    b = ProgramBuilder()
    grad_ops, gens = [], ""
    rows = 0
    for layer, order in enumerate(("XYZ", "ZYX")):
        for g in order:
            for q in rng.permutation(n):
                b.add({"X": RX, "Y": RY, "Z": RZ}[g], [int(q)], param=float(rng.uniform(-3, 3)))
                grad_ops.append(rows)
                gens += g
                rows += 1
            c, t = (int(x) for x in rng.choice(n, 2, replace=False))
            b.add(GENERAL, [c, t], n_ctrl=1, matrix=_rot(g, float(rng.uniform(-3, 3))))
            grad_ops.append(rows)
            gens += g
            rows += 1
        for q in range(n - 1):
            b.add(CZ, [q, q + 1], n_ctrl=1)
            rows += 1
    prog = b.program(n_qubits=n)
    terms, coeffs = random_pauli_terms(n, 5, rng)
    want, e_want = og.adjoint(prog, n, grad_ops, gens, terms, coeffs)
    options = [("tile_bits", tile), ("low_bits", low)] if tile else []
    got, e = engine_adjoint(prog, n, grad_ops, gens, terms, coeffs, dtype=dtype, options=options)
    assert abs(e - e_want) < tol
    assert np.abs(got - want).max() < tol
