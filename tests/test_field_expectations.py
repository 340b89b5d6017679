"""Expectations of Z strings and single-qubit X / Y letters, which take one kernel that keeps every sum of a
tile, against numpy and against the kernel of general Pauli strings (one two-letter flip sends a list there)."""

from contextlib import closing

import numpy as np
import pytest

from pyquafu_amd import _native
from tests.conftest import rand_state


def _oracle(psi, letters, qubits):
    idx = np.arange(psi.size)
    sign = np.ones(psi.size)
    flip = 0
    factor = 1.0 + 0.0j
    for c, q in zip(letters, qubits):
        bit = (idx >> q) & 1
        if c in "XY":
            flip |= 1 << q
        if c in "YZ":
            sign = sign * (1 - 2 * bit)
        if c == "Y":
            factor *= 1j  # Y |b> = i (-1)^b |1 - b>
    return float(np.real(np.sum(np.conj(psi[idx ^ flip]) * factor * sign * psi)))


def _terms(n, rng, strings):
    terms = [(c, [q]) for c in "XYZ" for q in range(n)]
    for _ in range(strings):
        k = int(rng.integers(1, n + 1))
        terms.append(("Z" * k, [int(q) for q in rng.choice(n, k, replace=False)]))
    order = rng.permutation(len(terms))
    return [terms[i] for i in order]


# 12 qubits fill one tile, below that it is padded; 13 leaves one qubit outside, 17 and 21 (22) take one
# and two (three) passes at complex128; the longer lists make two batches of 256
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,strings", [(1, 1), (2, 3), (5, 20), (11, 230), (12, 40), (13, 40), (17, 300), (21, 9), (22, 3)])
def test_field_terms(n, strings, dtype):
    rng = np.random.default_rng(100 * n + strings)
    psi = rand_state(n, rng)
    if dtype == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    terms = _terms(n, rng, strings)
    if n < 5:  # lists of up to 12 terms stay with the general kernel
        terms = terms * 8
    with closing(_native.DeviceState(n, dtype)) as dev:
        dev.load(psi)
        got = np.array(dev.expect(terms))
        general = np.array([dev.expect([t, ("XX", [0, 1])])[0] for t in terms[:24]]) if n > 1 else got[:0]
    assert np.all(np.isfinite(got))
    # sums of 2^n float64 products of a unit vector in a tree: log2 rounding growth, n eps each way
    tol = 4 * (n + 12) * np.finfo(np.float64).eps
    np.testing.assert_allclose(general, got[: len(general)], rtol=0, atol=tol)
    some = range(len(terms)) if n <= 13 else range(0, len(terms), max(1, len(terms) // 24))
    for i in some:
        assert abs(got[i] - _oracle(psi, *terms[i])) < tol, terms[i]


@pytest.mark.gpu
def test_field_terms_carry_nan_and_inf():
    n = 14
    psi = np.zeros(1 << n, dtype=np.complex128)
    psi[5] = np.nan
    with closing(_native.DeviceState(n, "c128")) as dev:
        dev.load(psi)
        assert np.all(np.isnan(dev.expect([(c, [q]) for c in "XYZ" for q in range(n)] + [("ZZ", [0, 13])])))
