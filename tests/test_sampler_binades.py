"""The sampler that tells each block's binade from sums in another order, on states whose running sum meets
powers of two in every awkward way, against the oracle's sequential sum."""

from contextlib import closing

import numpy as np
import pytest

from oracle.cpu import sample_on
from pyquafu_amd import _native
from tests.conftest import rand_state

pytestmark = pytest.mark.gpu


def _state(kind, n, rng):
    size = 1 << n
    i = np.arange(size)
    if kind == "uniform":  # every power of two is reached exactly, on a block's edge
        return np.full(size, 2.0 ** (-n / 2), complex)
    if kind == "thirds":  # the same rounding error at every step
        return np.sqrt(np.where(i % 3 == 0, 1.0, 2.0) / (1.7 * size)).astype(complex)
    if kind == "ghz":  # one half, then long nothing
        psi = np.zeros(size, complex)
        psi[0] = psi[-1] = np.sqrt(0.5)
        return psi
    if kind == "last":
        psi = np.zeros(size, complex)
        psi[-1] = 1.0
        return psi
    if kind == "tail":  # the sum creeps towards 1 within the margin, for many blocks
        return np.sqrt(2.0 ** (-50 * i / size) * 35.0 / size) * np.exp(1j * i)
    if kind == "far tail":  # terms below half an ulp of the sum
        return np.sqrt(np.where(i < 40, 1.0 / 40, 1e-19 / size)).astype(complex)
    if kind == "steep":  # three binades an element
        return np.sqrt(np.exp2(np.maximum(-900.0 + 3.0 * i, -2000.0) * (i < 300))).astype(complex)
    if kind == "creep":  # half of every term is rounded away: other sums cross 1, the sequential one does not
        psi = np.full(size, np.sqrt(1.49 * 2.0**-53), complex)
        psi[0] = np.sqrt(1.0 - 1.2 * size * 2.0**-53)
        return psi
    if kind == "inf":
        psi = rand_state(n, rng)
        psi[size // 2] = np.inf
        return psi
    return rand_state(n, rng)


# 5: one block; 10 to 12: a tile's remainder, one and two tiles; 15, 18: many; 21, 22: one and two groups
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("kind", ["uniform", "thirds", "ghz", "last", "tail", "far tail", "steep", "creep", "inf", "random"])
@pytest.mark.parametrize("n", [5, 10, 11, 12, 15, 18])
def test_block_ends(n, kind, dtype):
    _check(n, kind, dtype, 3000)


@pytest.mark.parametrize("kind", ["uniform", "tail", "random"])
@pytest.mark.parametrize("n", [21, 22])
def test_block_ends_of_groups(n, kind):
    _check(n, kind, "c128", 20000)


# up to 2^20 shots stay in pinned memory
@pytest.mark.parametrize("shots", [1, 2, 1024, 1 << 20, (1 << 20) + 1])
def test_shot_counts(shots):
    _check(13, "random", "c128", shots)


def _check(n, kind, dtype, shots):
    rng = np.random.Generator(np.random.PCG64(900 + n))
    with closing(_native.DeviceState(n, dtype)) as dev:
        dev.load(_state(kind, n, rng))
        psi = dev.store()
        with np.errstate(invalid="ignore", over="ignore"):
            cdf = np.cumsum(np.abs(psi) ** 2)
        finite = cdf[np.isfinite(cdf)]
        total = float(finite[-1])
        at = finite[rng.integers(0, finite.size, size=shots)]
        u = np.concatenate([rng.random(shots) * total * 1.001, at, np.nextafter(at, 0.0), np.nextafter(at, np.inf)])
        u = u[rng.permutation(u.size)[:shots]]
        assert np.array_equal(dev.sample(u), sample_on(psi, u))
