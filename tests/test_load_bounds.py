"""The loads of the lazy transforms and key products (fhe_amd/csrc/f64mod.h):
what beyond_lazy lets through unreduced is non-negative and at most 4q, every
lazy residue passes, and an inverse pass and a key product on the widest
values let through stay exact in doubles."""
import random

import pytest

from test_f64_bounds import held, product
from test_lazy_bounds import brev, ntt_prime, root


def beyond(v, q):
    return (v % (1 << 64)) >> 32 > (2 * q - 1) >> 32 or q < 1 << 31


@pytest.mark.parametrize("bits", [20, 31, 32, 40, 42, 54, 60, 61])
def test_range_let_through(bits):
    q = ntt_prime(bits, 1 << 13)
    rng = random.Random(bits)
    edge = [(2 * q - 1 | 0xffffffff) + d for d in (0, 1)]
    for v in edge + [0, 1, 2 * q - 1, -1, -q, 1 << 62, -(1 << 62)] + [
            rng.randrange(8 * q) for _ in range(2000)]:
        if not beyond(v, q):
            assert 0 <= v < 2 * q + (1 << 32) <= 4 * q
        elif q > 1 << 31:
            assert not 0 <= v < 2 * q


@pytest.mark.parametrize("bits", [32, 40, 42])
def test_widest_values_stay_exact(bits):
    n, q = 256, ntt_prime(bits, 1 << 14)
    top = 2 * q - 1 | 0xffffffff
    assert not beyond(top, q)
    psi = root(q, n)
    rng = random.Random(bits)
    start = [rng.choice((0, top)) - q for _ in range(n)]
    x, e = list(start), [v % q for v in start]
    for t in range(8):
        half = 1 << t
        for g in range(n // (2 * half)):
            w = pow(psi, -brev(n // (2 * half) + g, 8), q)
            for j in range(2 * g * half, 2 * g * half + half):
                a, b = x[j], x[j + half]
                x[j], x[j + half] = held(a + b), product(a - b, w, q)
                a, b = e[j], e[j + half]
                e[j], e[j + half] = (a + b) % q, (a - b) * w % q
    assert [v % q for v in x] == e
    # key products: own limbs load below 2^47 in magnitude
    for y in (1 << 47, -(1 << 47), 13 * q):
        if abs(y) <= 1 << 47:
            assert (product(y, top, q) - y * top) % q == 0
