"""N = 2^17, whose transforms run one 8-bit register pass and one generic
exact pass: key switching gives the limbs of the oracle.  There and on the
other rings, the key's stage of slot-to-coeff (attached input, full
decompositions, baby and giant steps) gives the same limbs with and without
lazy arithmetic."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu

ALPHA = 2


def is_prime(x):
    """Miller-Rabin with bases that decide every x below 2^64."""
    bases = (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37)
    if any(x % a == 0 for a in bases):
        return x in bases
    d, r = x - 1, 0
    while d % 2 == 0:
        d, r = d // 2, r + 1
    return all(pow(a, d, x) == 1 or
               any(pow(a, d << i, x) == x - 1 for i in range(r))
               for a in bases)


def primes_of(log_n, bits, count):
    """The `count` largest NTT primes below 2^bits for N = 2^log_n."""
    step = 2 << log_n
    x, out = (1 << bits) // step * step + 1, []
    while len(out) < count:
        x -= step
        assert x > 1, "no more primes"
        if is_prime(x):
            out.append(x)
    return out


def chain(log_n, bits):
    big = primes_of(log_n, 60, 2 + ALPHA)
    return np.array(big[:1] + primes_of(log_n, bits, 4) + big[1:], np.uint64)


def test_key_switching(gpu_lib):
    log_n = 17
    primes = chain(log_n, 40)
    rng = np.random.Generator(np.random.PCG64(17))
    with fhe_amd.Context(log_n, ALPHA, primes=primes) as ctx:
        n, key_mid = ctx.n, ctx.key_moduli_id()
        mid = key_mid
        limbs = ctx.limbs_at(mid)
        ct = uniform(rng, primes, mid, (2, limbs, n))
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid), 2)
        d, dk = ctx.to_device(ct[None]), ctx.to_device(key)
        out = ctx.array((1, 2, limbs, n))
        ctx.switch_key(d, dk, key_mid, out, mid)
        got = out.download()[0]
        for arr in (d, dk, out):
            arr.free()
    want = Oracle(log_n, primes, ALPHA).switch_key(ct, key, mid, key_mid)
    same = np.array_equal(got, want)
    assert same


@pytest.mark.parametrize("log_n,bits", [(11, 40), (13, 40), (14, 54), (15, 40),
                                        (16, 40), (16, 54), (17, 40),
                                        (17, 54)])
def test_key_stage_lazy_equals_exact(gpu_lib, log_n, bits):
    primes = chain(log_n, bits)
    rng = np.random.Generator(np.random.PCG64(18))
    with fhe_amd.Context(log_n, ALPHA, primes=primes) as ctx:
        n, full, key_mid = ctx.n, ctx.info["full_level"], ctx.key_moduli_id()
        level = full - 1
        mid = full - level + 1  # the stage's, rescaled
        made = []

        def dev(host):
            made.append(ctx.to_device(host))
            return made[-1]

        ext = ctx.limbs_at(mid) + ALPHA
        diagonal = np.concatenate([
            uniform(rng, primes, mid, (ctx.limbs_at(mid), n)),
            uniform(rng, primes, ctx.chain_count, (ALPHA, n))])
        assert diagonal.shape == (ext, n)
        diagonals = {(o, i): dev(diagonal) for o in (0, 1) for i in (0, 1)
                     if o or i}
        key = dev(uniform(rng, primes, key_mid, ctx.key_shape(key_mid)))
        stage = fhe_amd.PlainMatrix.make(level, [0, 1], [0, 2], diagonals)
        bk = ctx.bootstrap_key(fhe_amd.BootstrapKeyParts.make(
            [], [stage], [(1, key, key_mid), (2, key, key_mid)]))
        texts = [dev(uniform(rng, primes, full - level,
                             (1, 2, ctx.limbs_at(full - level), n)))
                 for _ in range(2)]
        got = []
        for lazy in (0, 1):
            ctx.set_option("lazy_key_switch", lazy)
            out = dev(np.zeros((1, 2, ctx.limbs_at(mid), n), np.int64))
            print(f"slot_to_coeff_bk N=2^{log_n} lazy {lazy}", flush=True)
            ctx.slot_to_coeff_bk(texts[0], texts[1], level, 0, key, key_mid,
                                 bk, out)
            got.append(out.download())
        ctx.set_option("lazy_key_switch", 1)
        ctx.bootstrap_key_destroy(bk)
        for arr in made:
            arr.free()
    assert np.count_nonzero(got[0]) > n
    same = np.array_equal(got[0], got[1])
    assert same
