"""Keys and NTT-form trios that are other representatives of their residues
give the limbs of the canonical ones: the double-held and lazy forms look at
the range of what they load.  Against the oracle, limb for limb."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu

CASES = [(13, 1, 3), (15, 2, 7), (16, 4, 6)]


def small(q):
    return q < 1 << 42


@pytest.mark.parametrize("log_n,alpha,limbs", CASES)
def test_wide_keys(gpu_lib, log_n, alpha, limbs):
    """Key residues of the primes below 2^42 up to 2^60."""
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(21))
    orc = Oracle(log_n, primes, alpha)
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        a = uniform(rng, primes, mid, (1, 2, limbs, n))
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid))
        wide = key.copy()
        for l in range(key.shape[1]):
            q = int(primes[key_mid + l])
            if small(q):
                # one coefficient in 64 wide, a polynomial wide throughout
                most = (1 << 60) // q
                wide[:, l, ::64] += q * rng.integers(0, most, n // 64)
                wide[-1, l] = key[-1, l] + q * rng.integers(0, most, n)
        da, dk = ctx.to_device(a), ctx.to_device(wide)
        rot = ctx.array((1, 2, limbs, n))
        out = ctx.array((1, 2, limbs - 1, n))
        print(f"wide keys N=2^{log_n}", flush=True)
        ctx.rotate(da, dk, key_mid, 3, rot, mid)
        ctx.hmult_relin_rescale(da, da, dk, key_mid, out, mid)
        got, prod = rot.download(), out.download()
        for arr in (da, dk, rot, out):
            arr.free()
    same = [np.array_equal(got[0], orc.rotate(a[0], key, mid, key_mid, 3)),
            np.array_equal(prod[0], orc.hmult(a[0], a[0], key, mid, key_mid))]
    assert same == [True, True]


@pytest.mark.parametrize("log_n,alpha,limbs", CASES)
def test_wide_trios(gpu_lib, log_n, alpha, limbs):
    """NTT-form trios: +-2^45 for primes below 2^42, [-q, 3q) for others."""
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(22))
    orc = Oracle(log_n, primes, alpha)
    count = 2
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        trios = uniform(rng, primes, mid, (count, 3, limbs, n))
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid))
        wide = trios.copy()
        for l in range(limbs):
            q = int(primes[mid + l])
            most = (1 << 45) // q
            lo, hi = (-most, most) if small(q) else (-1, 3)
            # ciphertext 0 wide throughout, 1 in one coefficient of 1024
            wide[0, :, l] += q * rng.integers(lo, hi, (3, n))
            wide[1, :, l, ::1024] += q * rng.integers(lo, hi, (3, n // 1024))
        dt, dk = ctx.to_device(wide), ctx.to_device(key)
        out = ctx.array((count, 2, limbs, n))
        print(f"wide trios N=2^{log_n}", flush=True)
        ctx.relinearize(dt, dk, key_mid, out, mid)
        got = out.download()
        if log_n == 16:
            each = [ctx.to_device(t) for t in wide]
            outs = [ctx.array((2, limbs, n)) for _ in each]
            ctx.relinearize_uneven(each, [mid] * count, dk, key_mid, outs)
            uneven = [o.download() for o in outs]
            for arr in each + outs:
                arr.free()
        for arr in (dt, dk, out):
            arr.free()
    if log_n == 16:
        assert [np.array_equal(u, g) for u, g in zip(uneven, got)] == \
            [True] * count
    same = [np.array_equal(got[c], orc.relinearize(trios[c], key, mid,
                                                   key_mid))
            for c in range(count)]
    assert same == [True] * count
