"""fhe_multiply with a relinearization key against the exact trio product
followed by fhe_relinearize, limb for limb, on every pair of input forms: the
two transform the factors differently (lazily from the coefficient domain, or
exactly into the returned trio)."""
import itertools

import numpy as np
import pytest

import fhe_amd
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu

NTT, RESCALED = fhe_amd.FLAG_NTT_FORM, fhe_amd.FLAG_RESCALED
FORMS = [(level, flags) for level in (5, 4)
         for flags in (0, RESCALED, NTT, NTT | RESCALED)]


@pytest.mark.parametrize("log_n,alpha", [(14, 1), (16, 4)])
def test_forms(gpu_lib, log_n, alpha):
    count = 2
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, full = ctx.n, ctx.info["full_level"]
        key_mid = ctx.key_moduli_id()
        rng = np.random.Generator(np.random.PCG64(5))
        key = ctx.to_device(uniform(rng, ctx.primes, key_mid,
                                    ctx.key_shape(key_mid), 2))
        texts = {}
        for level, flags in FORMS:
            mid = full - level + (1 if flags & RESCALED else 0)
            texts[level, flags] = ctx.to_device(uniform(
                rng, ctx.primes, mid, (count, 2, ctx.limbs_at(mid), n)))
        pairs = list(itertools.product(FORMS, FORMS)) if log_n == 14 else [
            ((5, 0), (5, 0)), ((5, NTT | RESCALED), (5, RESCALED)),
            ((4, RESCALED), (4, RESCALED)), ((5, NTT), (4, NTT | RESCALED))]
        for (la, fa), (lb, fb) in pairs:
            mid = full - min(la, lb) + 1
            limbs = ctx.limbs_at(mid)
            trio = ctx.array((count, 3, limbs, n))
            want = ctx.array((count, 2, limbs, n))
            got = ctx.array((count, 2, limbs, n))
            a, b = texts[la, fa], texts[lb, fb]
            ctx.multiply(a, la, fa, b, lb, fb, trio)
            ctx.relinearize(trio, key, key_mid, want, mid)
            ctx.multiply(a, la, fa, b, lb, fb, got, key, key_mid)
            assert np.array_equal(got.download(), want.download()), (
                la, fa, lb, fb)
            for arr in (trio, want, got):
                arr.free()
        for arr in [key] + list(texts.values()):
            arr.free()


@pytest.mark.parametrize("log_n,alpha,shift", [(13, 1, 0), (14, 1, 1),
                                               (15, 2, 0)])
def test_batches_equal_single_texts(gpu_lib, log_n, alpha, shift):
    """Plaintext products, encryption and decryption of a batch against each
    text alone; shift: operands 8 bytes past a 16-byte boundary."""
    count, level = 3, 2
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, full = ctx.n, ctx.info["full_level"]
        rng = np.random.Generator(np.random.PCG64(6))
        mid = full - level
        limbs = ctx.limbs_at(mid)
        made = []

        class At:
            """A device array of `shape` starting `shift` words in."""

            def __init__(self, shape, host=None):
                whole = ctx.array((int(np.prod(shape)) + 2,))
                made.append(whole)
                self.whole, self.shape = whole, shape
                self.ptr = type(whole.ptr)(whole.ptr.value + 8 * shift)
                if host is not None:
                    whole.upload_at(np.ascontiguousarray(host), shift)

            def download(self):
                flat = self.whole.download()
                return flat[shift:shift + int(np.prod(self.shape))].reshape(
                    self.shape)

        ct = uniform(rng, ctx.primes, mid, (count, 2, limbs, n))
        pt = uniform(rng, ctx.primes, mid, (count, limbs, n))
        keys = uniform(rng, ctx.primes, 0, (2, ctx.chain_count, n))
        small = rng.integers(-4, 5, (3, count, n))

        def run(sel):
            k = len(sel)
            c, p = At((k, 2, limbs, n), ct[sel]), At((k, limbs, n), pt[sel])
            pk, sk = At(keys.shape, keys), At(keys.shape[1:], keys[0])
            u, e0, e1 = (At((k, n), x[sel]) for x in small)
            prod = At((k, 2, limbs - 1, n))
            enc, dec = At((k, 2, limbs, n)), At((k, limbs, n))
            ctx.multiply_plain(c, level, 0, p, level, 0, prod)
            ctx.encrypt_pk(p, pk, 0, u, e0, e1, enc, mid)
            ctx.decrypt(c, sk, 0, dec, mid)
            return [x.download() for x in (prod, enc, dec)]

        whole = run(list(range(count)))
        for i in range(count):
            for w, one in zip(whole, run([i])):
                assert np.array_equal(w[i], one[0])
        for arr in made:
            arr.free()
