"""Key switching on the rings below N = 2^16, whose transforms run in passes
of 6 to 8 bits and whose key switching holds every partition at once: HMult +
relinearize + rescale, rotation and the allocation-free entry point against
the oracle, limb for limb, at full and ragged partitions of 1 to 8 limbs."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle

pytestmark = pytest.mark.gpu

# (log N, special primes, limbs): one-limb partitions, partitions of 2, 3
# and 5 limbs with a shorter first one, and the eight-limb form; the lowest
# level and the top one of each chain
CASES = [(13, 1, 3), (14, 1, 8), (14, 1, 3), (14, 3, 5), (15, 2, 17),
         (15, 5, 11), (15, 8, 9), (15, 8, 3)]


def uniform(rng, primes, mid, shape, factor=1):
    limbs, n = shape[-2:]
    out = np.empty(shape, np.int64)
    for l in range(limbs):
        out[..., l, :] = rng.integers(0, int(primes[mid + l]) * factor,
                                      shape[:-2] + (n,), dtype=np.uint64)
    return out


@pytest.mark.parametrize("log_n,alpha,limbs", CASES)
def test_key_switching(gpu_lib, log_n, alpha, limbs):
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(log_n * 100 + alpha + limbs))
    orc = Oracle(log_n, primes, alpha)
    count = 2
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        a = uniform(rng, primes, mid, (count, 2, limbs, n))
        b = uniform(rng, primes, mid, (count, 2, limbs, n))
        a[0, :, :, ::7] = 0  # zero residues beside random ones
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid), 2)
        da, db, dk = (ctx.to_device(x) for x in (a, b, key))
        out = ctx.array((count, 2, limbs - 1, n))
        again = ctx.array((count, 2, limbs - 1, n))
        rot = ctx.array((count, 2, limbs, n))
        print(f"N=2^{log_n} alpha {alpha} limbs {limbs}", flush=True)
        ctx.hmult_relin_rescale(da, db, dk, key_mid, out, mid)
        got = out.download()
        assert fhe_amd.library().fhe_hmult_relin_rescale_noalloc(
            ctx.handle, count, mid, da.ptr, db.ptr, dk.ptr, key_mid,
            again.ptr) == 0
        assert np.array_equal(again.download(), got)
        ctx.rotate(da, dk, key_mid, 3, rot, mid)
        rotated = rot.download()
        for arr in (da, db, dk, out, again, rot):
            arr.free()
    for c in range(count):
        assert np.array_equal(got[c], orc.hmult(a[c], b[c], key, mid,
                                                key_mid)), c
        assert np.array_equal(rotated[c], orc.rotate(a[c], key, mid, key_mid,
                                                     3)), c


def test_noalloc_splits_batches(gpu_lib):
    """A batch whose fused workspace exceeds the fixed scratch (105 MB a pair
    at N = 2^15, 18 limbs) runs in parts, with the same limbs."""
    with fhe_amd.Context(15, 2) as ctx:
        n, limbs, count = ctx.n, 18, 7
        mid, key_mid = ctx.chain_count - limbs, ctx.key_moduli_id()
        rng = np.random.Generator(np.random.PCG64(3))
        a = uniform(rng, ctx.primes, mid, (count, 2, limbs, n))
        key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
        da, dk = ctx.to_device(a), ctx.to_device(key)
        want = ctx.array((count, 2, limbs - 1, n))
        got = ctx.array((count, 2, limbs - 1, n))
        ctx.hmult_relin_rescale(da, da, dk, key_mid, want, mid)
        assert fhe_amd.library().fhe_hmult_relin_rescale_noalloc(
            ctx.handle, count, mid, da.ptr, da.ptr, dk.ptr, key_mid,
            got.ptr) == 0
        assert np.array_equal(want.download(), got.download())
        for arr in (da, dk, want, got):
            arr.free()


@pytest.mark.parametrize("log_n,alpha,limbs", [(13, 1, 3), (16, 4, 6)])
def test_wild_representatives(gpu_lib, log_n, alpha, limbs):
    """Inputs that are other representatives of their residues, up to 2^61 in
    magnitude (the load of the double-held transforms and of the first
    digits): polynomial 0 of the factors of a product, and a rotation."""
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(9))
    orc = Oracle(log_n, primes, alpha)
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        a = uniform(rng, primes, mid, (1, 2, limbs, n))
        b = uniform(rng, primes, mid, (1, 2, limbs, n))
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid), 2)
        wild = a.copy()
        for l in range(limbs):
            q = int(primes[mid + l])
            if q < 1 << 42:
                most = (1 << 61) // q
                wild[0, 0, l] += q * rng.integers(-most, most, n)
        da, db, dk = (ctx.to_device(x) for x in (wild, b, key))
        out = ctx.array((1, 2, limbs - 1, n))
        ctx.hmult_relin_rescale(da, db, dk, key_mid, out, mid)
        got = out.download()
        for arr in (da, db, dk, out):
            arr.free()
    assert np.array_equal(got[0], orc.hmult(a[0], b[0], key, mid, key_mid))
