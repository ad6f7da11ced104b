"""HMult + relinearize + rescale of factors with values in (-q, q) on the
primes below 2^42, as rescaling by a 60-bit prime leaves them, or in
(-2^60, 2^60): dense ones (the lazy transforms), and sparse ones, whose
products have limbs with zero residues that are recomputed from the signed
values exactly.  Against the oracle, limb for limb, under each transform
arithmetic."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_small_rings import uniform
from test_gpu_zero_residues import sparse

pytestmark = pytest.mark.gpu


def negate_some(rng, primes, mid, x):
    """Other representatives x - q of about half the nonzero values."""
    for l in range(x.shape[-2]):
        q = int(primes[mid + l])
        if q < 1 << 42:
            v = x[..., l, :]
            v -= q * (rng.integers(0, 2, v.shape) & (v != 0))
    return x


def wide(rng, primes, mid, x):
    """Other representatives of the nonzero values, up to 2^60."""
    for l in range(x.shape[-2]):
        q = int(primes[mid + l])
        if q < 1 << 42:
            v, most = x[..., l, :], (1 << 60) // q
            v += q * (rng.integers(-most, most, v.shape) * (v != 0))


@pytest.mark.parametrize("log_n,alpha,limbs", [(13, 1, 3), (14, 1, 4),
                                               (15, 2, 5), (16, 4, 6)])
def test_signed_products(gpu_lib, log_n, alpha, limbs):
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(30 + log_n))
    orc = Oracle(log_n, primes, alpha)
    count = 4
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        a = uniform(rng, primes, mid, (count, 2, limbs, n))
        b = uniform(rng, primes, mid, (count, 2, limbs, n))
        for c, terms in ((1, 1), (2, 3), (3, 3)):
            a[c, 1] = sparse(rng, primes, mid, (limbs, n), terms)
            b[c, 1] = sparse(rng, primes, mid, (limbs, n), terms)
        a, b = (negate_some(rng, primes, mid, x) for x in (a, b))
        wide(rng, primes, mid, a[3])
        wide(rng, primes, mid, b[3])
        # constants that enter the Montgomery form as -1: the only way that
        # a negative value reaches the end of the exact transform (a
        # butterfly adds to the upper value, and its products are positive)
        for l in range(limbs):
            q = int(primes[mid + l])
            if q < 1 << 42:
                a[1, 1, l] = 0
                a[1, 1, l, 0] = a[3, 1, l, 0] = -pow(1 << 62, -1, q)
                b[2, 1, l] = 0
                b[2, 1, l, 0] = -pow(1 << 62, -1, q)
        assert (a < 0).any() and (b[2, 1] < 0).any()
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid), 2)
        da, db, dk = (ctx.to_device(x) for x in (a, b, key))
        out = ctx.array((count, 2, limbs - 1, n))
        got = []
        for lazy in (1, 0):
            print(f"signed N=2^{log_n} lazy {lazy}", flush=True)
            ctx.set_option("lazy_key_switch", lazy)
            ctx.hmult_relin_rescale(da, db, dk, key_mid, out, mid)
            got.append(out.download())
        for arr in (da, db, dk, out):
            arr.free()
    for c in range(count):
        want = orc.hmult(a[c], b[c], key, mid, key_mid)
        for lazy in (1, 0):
            same = np.array_equal(got[1 - lazy][c], want)
            assert same, (c, lazy)


@pytest.mark.parametrize("log_n,alpha", [(13, 1), (14, 2), (16, 4)])
def test_signed_values_elsewhere(gpu_lib, log_n, alpha):
    """Transforms, decryption and key switching of values in (-q, q)."""
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(60 + log_n))
    orc = Oracle(log_n, primes, alpha)
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid = ctx.n, 1
        limbs, key_mid = ctx.limbs_at(mid), ctx.key_moduli_id()
        x = negate_some(rng, primes, mid,
                        uniform(rng, primes, mid, (2, limbs, n)))
        assert (x < 0).any()
        same = []
        for enter in (True, False):
            d = ctx.to_device(x)
            ctx.ntt(d, mid, enter=enter)
            y = d.download()
            same.append(np.array_equal(y, orc.ntt(x, mid, enter=enter)))
            d.free()
        for z in (y, x):
            d = ctx.to_device(z)
            ctx.intt(d, mid, post=1)
            same.append(np.array_equal(d.download(), orc.intt(z, mid, post=1)))
            d.free()
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid))
        sk = uniform(rng, primes, 0, (ctx.chain_count, n))
        dx, dk, ds = (ctx.to_device(v) for v in (x[None], key, sk))
        pt, out = ctx.array((1, limbs, n)), ctx.array((1, 2, limbs, n))
        ctx.decrypt(dx, ds, 0, pt, mid)
        ctx.switch_key(dx, dk, key_mid, out, mid)
        same.append(np.array_equal(pt.download()[0],
                                   orc.decrypt(x, sk, 0, mid)))
        same.append(np.array_equal(out.download()[0],
                                   orc.switch_key(x, key, mid, key_mid)))
        for arr in (dx, dk, ds, pt, out):
            arr.free()
    assert same == [True] * 6
