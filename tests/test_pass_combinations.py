"""Which arithmetics the two passes of a forward transform may have
(fhe_amd/csrc/ntt.hip launch_r16_pass), in a model with 64-bit wrap-around:
exact after exact and lazy after lazy (kLazyLarge, settled at the end) give
the transform's residues for inputs up to the extension's 4q; the exact
butterflies after a lazy pass do not for 60-bit primes, which is why the
8-bit pass of N = 2^17, whose other pass is the generic exact kernel, runs
exact too."""
import random

import pytest

from test_lazy_bounds import brev, ntt_prime, root

M64 = (1 << 64) - 1
LOG_N, FIRST = 10, 8


def signed(x):
    x &= M64
    return x - (1 << 64) if x >> 63 else x


def mont(a, b, q, k):
    """The unsigned Montgomery product of 64-bit words (mont_mult_u), of
    b + 2^62 in place of b for a signed operand (mont_mult_cs)."""
    b = (b + (1 << 62)) & M64
    x = a * b
    s = (x * k) & ((1 << 62) - 1)
    return signed(((x + s * q) >> 62) - a)


def guard(x, m):
    return x - m if x >= m else x


def exact(x, y, w, q, k):
    p = mont(w * (1 << 62) % q, y, q, k)
    return (guard(signed(x + p), 2 * q), guard(signed(x + 2 * q - p), 2 * q))


def lazy(x, y, w, q, _):
    wq = (w << 64) // q
    y0, y1, v0, v1 = y & 0xffffffff, y >> 32, wq & 0xffffffff, wq >> 32
    h = v1 * y1 + (v0 * y1 >> 32) + (v1 * y0 >> 32)
    p = (w * y - h * q) & M64
    x = guard(x, 4 * q)
    return (x + p) & M64, (x + 4 * q - p) & M64


def transform(start, q, psi, passes):
    n, k = 1 << LOG_N, -pow(q, -1, 1 << 62) % (1 << 62)
    x, want = list(start), [v % q for v in start]
    for s in range(LOG_N):
        half = n >> (s + 1)
        step = passes[0 if s < FIRST else 1]
        for g in range(1 << s):
            w = pow(psi, brev((1 << s) + g, LOG_N), q)
            for j in range(2 * g * half, 2 * g * half + half):
                x[j], x[j + half] = step(x[j], x[j + half], w, q, k)
                p = want[j + half] * w % q
                want[j], want[j + half] = want[j] + p, want[j] - p
    return sum((a - b) % q != 0 for a, b in zip(x, want))


@pytest.mark.parametrize("passes,bits,sound", [
    ((exact, exact), 54, True), ((exact, exact), 60, True),
    ((lazy, lazy), 54, True), ((lazy, lazy), 60, True),
    ((lazy, exact), 54, True), ((lazy, exact), 60, False)])
def test_pass_combinations(passes, bits, sound):
    q = ntt_prime(bits, 1 << 17)
    rng = random.Random(bits)
    top = 2 * q if passes[0] is exact else 4 * q
    start = [top - 1 - rng.randrange(1 << 40) for _ in range(1 << LOG_N)]
    wrong = transform(start, q, root(q, 1 << LOG_N), passes)
    assert (wrong == 0) == sound, wrong
