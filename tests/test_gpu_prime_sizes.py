"""Explicit chains whose primes lie at the edges of the arithmetics: just
below and above 2^42 (doubles or 64-bit integers), around 2^31 (below it every
load is reduced), 18 to 24 bits, and special primes just below 2^61.  (Products
of two lazy residues need q <= 2^60: chain primes stay below that, and keys
below q.)  HMult + relinearize + rescale, rotation and relinearization against
the oracle, limb for limb."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_large_ring import primes_of
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n,alpha,bits", [
    (13, 1, (60, 42, 42, 31, 32, 18, 60, 60)),
    (14, 2, (60, 42, 43, 30, 41, 24, 60, 61, 61)),
    (15, 2, (60, 42, 20, 42, 33, 54, 60, 61, 61)),
    (16, 3, (60, 42, 20, 31, 43, 42, 60, 61, 61, 61))])
def test_prime_sizes(gpu_lib, log_n, alpha, bits):
    # the k-th largest prime of its size for the k-th of that size
    primes = np.array([primes_of(log_n, b, bits[:i].count(b) + 1)[-1]
                       for i, b in enumerate(bits)], np.uint64)
    assert len(set(primes.tolist())) == len(bits)
    rng = np.random.Generator(np.random.PCG64(70))
    orc = Oracle(log_n, primes, alpha)
    with fhe_amd.Context(log_n, alpha, primes=primes) as ctx:
        n, mid, key_mid = ctx.n, ctx.key_moduli_id(), ctx.key_moduli_id()
        limbs = ctx.limbs_at(mid)
        a, b = (uniform(rng, primes, mid, (2, 2, limbs, n)) for _ in range(2))
        a[1, :, :, ::3] = 0
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid))
        trios = uniform(rng, primes, mid, (2, 3, limbs, n))
        da, db, dk, dt = (ctx.to_device(x) for x in (a, b, key, trios))
        out = ctx.array((2, 2, limbs - 1, n))
        rot, rel = (ctx.array((2, 2, limbs, n)) for _ in range(2))
        got = []
        for lazy in (1, 0):
            print(f"N=2^{log_n} primes of {bits} bits, lazy {lazy}",
                  flush=True)
            ctx.set_option("lazy_key_switch", lazy)
            ctx.hmult_relin_rescale(da, db, dk, key_mid, out, mid)
            ctx.rotate(da, dk, key_mid, 3, rot, mid)
            ctx.relinearize(dt, dk, key_mid, rel, mid)
            got.append([x.download() for x in (out, rot, rel)])
        for arr in (da, db, dk, dt, out, rot, rel):
            arr.free()
    for c in range(2):
        want = (orc.hmult(a[c], b[c], key, mid, key_mid),
                orc.rotate(a[c], key, mid, key_mid, 3),
                orc.relinearize(trios[c], key, mid, key_mid))
        same = [[np.array_equal(x[c], w) for x, w in zip(g, want)]
                for g in got]
        assert same == [[True] * 3] * 2, c
