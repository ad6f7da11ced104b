"""The 64-bit lazy butterflies with the short Shoup quotient
(fhe_amd/csrc/modarith.h shoup_short, ntt_r16.h kLazyLarge) in exact
integers: the quotient misses at most two, so products lie in [0, 4q), forward
values in [0, 8q) and inverse values in [0, 4q) for every q < 2^61, without
64-bit wrap-around, and the residues are the transform's."""
import random

import pytest

from test_lazy_bounds import brev, ntt_prime, root

M64 = (1 << 64) - 1


def shoup_short(y, w, q):
    assert 0 <= y <= M64
    wq = (w << 64) // q
    y0, y1, v0, v1 = y & 0xffffffff, y >> 32, wq & 0xffffffff, wq >> 32
    h = v1 * y1 + (v0 * y1 >> 32) + (v1 * y0 >> 32)
    assert 0 <= (wq * y >> 64) - h <= 2
    r = (w * y - h * q) & M64
    assert r == w * y - h * q and r < 4 * q
    return r


def guard(x, m):
    assert 0 <= x <= M64
    return x - m if x >= m else x


@pytest.mark.parametrize("bits", [43, 54, 60, 61])
def test_short_quotient_transforms(bits):
    n = 256
    q = ntt_prime(bits, 1 << 14)
    assert q < 1 << 61
    psi = root(q, n)
    rng = random.Random(bits)
    start = [rng.choice((2 * q - 1, 0, q, rng.randrange(2 * q)))
             for _ in range(n)]
    x, e = list(start), [v % q for v in start]
    for s in range(8):
        half = n >> (s + 1)
        for g in range(1 << s):
            w = pow(psi, brev((1 << s) + g, 8), q)
            for j in range(2 * g * half, 2 * g * half + half):
                k = j + half
                p, a = shoup_short(x[k], w, q), guard(x[j], 4 * q)
                x[j], x[k] = a + p, a + 4 * q - p
                assert max(x[j], x[k]) < min(8 * q, 1 << 64)
                pe = e[k] * w % q
                e[j], e[k] = (e[j] + pe) % q, (e[j] - pe) % q
    assert [v % q for v in x] == e
    settled = [guard(guard(v, 4 * q), 2 * q) for v in x]
    assert max(settled) < 2 * q
    x = settled
    for t in range(8):
        half = 1 << t
        for g in range(n // (2 * half)):
            w = pow(psi, -brev(n // (2 * half) + g, 8), q)
            for j in range(2 * g * half, 2 * g * half + half):
                k = j + half
                a, b = x[j], x[k]
                x[j] = guard(a + b, 4 * q)
                x[k] = shoup_short(a + 4 * q - b, w, q)
                assert max(x[j], x[k]) < 4 * q
    inv = pow(n, -1, q)
    assert [v * inv % q for v in x] == [v % q for v in start]


def test_extension_sum():
    """Sums of short products with one guard of 4q a term stay below 4q."""
    rng = random.Random(1)
    for bits in (54, 60, 61):
        q = ntt_prime(bits, 1 << 14)
        for _ in range(200):
            y, want = 0, 0
            for j in range(16):
                d, c = rng.randrange(1 << 62), rng.randrange(q)
                y += shoup_short(d, c, q)
                y = guard(y, 4 * q) if j else y
                want = (want + d * c) % q
                assert y < 4 * q and y % q == want
