"""States for which sums in another order do not tell every block's binade: the sampler's chunk loop goes on from
the first block concerned. Against the oracle's sequential sum."""

from contextlib import closing

import numpy as np
import pytest

from oracle.cpu import sample_on
from pyquafu_amd import _native
from tests.conftest import rand_state

pytestmark = pytest.mark.gpu


def _check(psi, dtype, rng, shots=3000):
    n = int(psi.size).bit_length() - 1
    with closing(_native.DeviceState(n, dtype)) as dev:
        dev.load(psi)
        psi = dev.store()
        with np.errstate(invalid="ignore", over="ignore"):
            cdf = np.cumsum(np.abs(psi) ** 2)
        finite = cdf[np.isfinite(cdf)]
        total = float(finite[-1]) if finite.size else 1.0
        u = rng.random(shots) * total * 1.001
        if finite.size:
            at = finite[rng.integers(0, finite.size, size=shots)]
            u = np.concatenate([u, at, np.nextafter(at, 0.0), np.nextafter(at, np.inf)])
        u = u[rng.permutation(u.size)[:shots]]
        assert np.array_equal(dev.sample(u), sample_on(psi, u))


# one amplitude of nearly 1 among equal ones: their roundings are all the same, and many blocks lie within the
# margin of 1 (more than are replayed)
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("k", range(4, 12))
@pytest.mark.parametrize("n,where", [(16, 0.3), (20, 0.0), (20, 0.6), (21, 0.3)])
def test_equal_tails(n, where, k, dtype):
    rng = np.random.Generator(np.random.PCG64(60 * n + k))
    size = 1 << n
    psi = np.full(size, np.sqrt(10.0**-k / size), complex)
    psi[int(where * size)] = np.sqrt(1 - 10.0**-k)
    _check(psi, dtype, rng)


# (more shots than pinned memory holds are in the scratch behind the ends)
def test_shots_beyond_pinned_memory():
    rng = np.random.Generator(np.random.PCG64(9))
    size = 1 << 20
    psi = np.full(size, np.sqrt(1e-8 / size), complex)
    psi[size // 3] = np.sqrt(1 - 1e-8)
    _check(psi, "c128", rng, (1 << 20) + 5)


@pytest.mark.parametrize("at", [0, 1, 31, 32, 2047, 2048, 70000, (1 << 18) - 1])
@pytest.mark.parametrize("zeros", [0, 5000])
def test_infinite_from_any_block(zeros, at):
    n = 18
    rng = np.random.Generator(np.random.PCG64(at))
    psi = rand_state(n, rng)
    psi[:zeros] = 0.0
    psi[at] = np.inf
    _check(psi, "c128", rng)


# sums that start below the smallest binade of a pair, then cross many
@pytest.mark.parametrize("n", [12, 16, 20])
def test_tiny_starts(n):
    rng = np.random.Generator(np.random.PCG64(n))
    size = 1 << n
    psi = np.sqrt(np.exp2(np.linspace(-1040, -1, size))) * np.exp(1j * rng.uniform(0, 6, size))
    _check(psi, "c128", rng)
