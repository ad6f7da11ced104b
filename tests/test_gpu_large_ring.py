"""N = 2^17, whose transforms run one 8-bit register pass and one generic
exact pass: the key's stage of slot-to-coeff (attached input, full
decompositions, baby and giant steps) and key switching give the same limbs
with and without lazy arithmetic, and key switching those of the oracle."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu

LOG_N, ALPHA = 17, 2


def primes_of(bits, count):
    """The `count` largest NTT primes of `bits` bits for N = 2^17."""
    step = 2 << LOG_N
    x, out = (1 << bits) // step * step + 1, []
    while len(out) < count:
        x -= step
        if all(pow(a, x - 1, x) == 1 for a in (2, 3, 5, 7)):
            out.append(x)
    return out


def chain():
    big = primes_of(60, 2 + ALPHA)
    return np.array(big[:1] + primes_of(40, 4) + big[1:], np.uint64)


def test_key_switching(gpu_lib):
    primes = chain()
    rng = np.random.Generator(np.random.PCG64(17))
    with fhe_amd.Context(LOG_N, ALPHA, primes=primes) as ctx:
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
    want = Oracle(LOG_N, primes, ALPHA).switch_key(ct, key, mid, key_mid)
    same = np.array_equal(got, want)
    assert same


def test_key_stage_lazy_equals_exact(gpu_lib):
    primes = chain()
    rng = np.random.Generator(np.random.PCG64(18))
    with fhe_amd.Context(LOG_N, ALPHA, primes=primes) as ctx:
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
            print(f"slot_to_coeff_bk N=2^17 lazy {lazy}", flush=True)
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
