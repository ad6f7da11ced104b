"""The exactness claims of the double-held modular arithmetic
(fhe_amd/csrc/f64mod.h), in a model that rounds every operation to the nearest
double: the product of worst-case operands is the exact integer y w - t q
below 0.875 q (0.55 q for |y| <= 2^47), every value that the device holds in
a double is an integer below 2^53, and sixteen forward stages and two passes
of eight inverse stages stay inside the stated bounds."""
import random

import pytest

from test_lazy_bounds import brev, ntt_prime, root


def fl(x):
    """The nearest double of an exact integer, as an integer."""
    return int(float(x))


def held(x):
    assert abs(x) < 1 << 53 and fl(x) == x
    return x


def product(y, w, q):
    held(y)
    h = fl(y * w)
    l = y * w - h
    assert fl(l) == l  # the fused multiply-add's error term
    t = round(float(h) * (1.0 / float(q)))  # to even, as rint
    held(t)
    return held(held(h - t * q) + l)


def primes(bits, n):
    return [ntt_prime(b, n) for b in bits]


@pytest.mark.parametrize("q", primes((30, 39, 40, 41, 42), 1 << 14))
def test_product_bounds(q):
    assert q < 1 << 42
    rng = random.Random(q)
    for top, bound in ((1 << 47, 0.55), (1 << 50, 0.875)):
        for _ in range(4000):
            y = rng.choice((top, -top, rng.randint(-top, top),
                            rng.randint(-q, q)))
            w = rng.choice((q - 1, q // 2, q // 2 + 1, rng.randrange(q)))
            r = product(y, w, q)
            assert (r - y * w) % q == 0
            assert abs(r) < bound * q + 1


@pytest.mark.parametrize("q", primes((40, 42), 1 << 14))
def test_floor_and_center(q):
    rng = random.Random(q)
    qi = 1.0 / float(q)
    for _ in range(4000):
        x = rng.choice((rng.randint(-1 << 50, 1 << 50),
                        q * rng.randint(-200, 200) + rng.randint(-2, 2)))
        f = held(x - int(float(x) * qi // 1) * q)
        assert 0 <= f <= q and (f - x) % q == 0
        c = held(x - round(float(x) * qi) * q)
        assert abs(c) <= q / 2 + 2 and (c - x) % q == 0


@pytest.mark.parametrize("bits", [40, 42])
def test_transform_bounds(bits):
    """Alternating worst-case inputs through 16 forward stages, and through
    two inverse passes of 8 stages from centred lazy residues, one
    2^8-point sub-transform a pass: the values and the residues."""
    n = 256
    q = ntt_prime(bits, 1 << 14)
    psi = root(q, n)
    rng = random.Random(bits)
    start = [rng.choice((2 * q - 1, 0, rng.randrange(2 * q)))
             for _ in range(n)]

    def forward(x, exact):
        for s in range(8):
            half = n >> (s + 1)
            for g in range(1 << s):
                w = pow(psi, brev((1 << s) + g, 8), q)
                for j in range(2 * g * half, 2 * g * half + half):
                    p = x[j + half] * w % q if exact else product(
                        x[j + half], w, q)
                    a = x[j]
                    x[j], x[j + half] = a + p, a - p
                    if not exact:
                        held(x[j]), held(x[j + half])
        return x

    def inverse(x, exact):
        for t in range(8):
            half = 1 << t
            for g in range(n // (2 * half)):
                w = pow(psi, -brev(n // (2 * half) + g, 8), q)
                for j in range(2 * g * half, 2 * g * half + half):
                    a, b = x[j], x[j + half]
                    x[j] = a + b
                    x[j + half] = ((a - b) * w % q if exact
                                   else product(a - b, w, q))
                    if not exact:
                        held(x[j])
        return x

    f = forward(forward(list(start), False), False)
    want = forward(forward(list(start), True), True)
    assert all((a - b) % q == 0 for a, b in zip(f, want))
    assert max(map(abs, f)) < 2 * q + 16 * 0.55 * q
    i = inverse([v - q for v in start], False)
    assert max(map(abs, i)) <= 1 << 50
    i = inverse([held(v - round(float(v) / float(q)) * q) for v in i], False)
    want = inverse(inverse(list(start), True), True)
    assert all((a - b) % q == 0 for a, b in zip(i, want))
