"""Zero residues of the inverse transform that feeds ModUp: their
representative, 0 or q, depends on the exact transform's history, so limbs
with one are recomputed exactly.  Products and relinearizations of sparse
polynomials (nearly every coefficient a zero residue) and of zero ones,
against the oracle, limb for limb."""
import numpy as np
import pytest

import fhe_amd
from support import Oracle
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu


def sparse(rng, primes, mid, shape, terms):
    out = np.zeros(shape, np.int64)
    for l in range(shape[-2]):
        q = int(primes[mid + l])
        for at in rng.integers(0, shape[-1], terms):
            out[..., l, at] = rng.integers(1, q)
    return out


@pytest.mark.parametrize("log_n,alpha,limbs", [(13, 1, 3), (14, 1, 4),
                                               (15, 2, 5), (16, 4, 6)])
def test_sparse_products(gpu_lib, log_n, alpha, limbs):
    primes = fhe_amd.resolve_primes(log_n, alpha)
    rng = np.random.Generator(np.random.PCG64(log_n))
    orc = Oracle(log_n, primes, alpha)
    count = 4
    with fhe_amd.Context(log_n, alpha) as ctx:
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        a = uniform(rng, primes, mid, (count, 2, limbs, n))
        b = uniform(rng, primes, mid, (count, 2, limbs, n))
        a[0, 1] = sparse(rng, primes, mid, (limbs, n), 1)
        b[0, 1] = sparse(rng, primes, mid, (limbs, n), 2)
        a[1, 1] = sparse(rng, primes, mid, (limbs, n), 3)
        b[1, 1] = sparse(rng, primes, mid, (limbs, n), 3)
        a[2, 1] = 0
        key = uniform(rng, primes, key_mid, ctx.key_shape(key_mid), 2)
        da, db, dk = (ctx.to_device(x) for x in (a, b, key))
        out = ctx.array((count, 2, limbs - 1, n))
        print(f"sparse N=2^{log_n}", flush=True)
        ctx.hmult_relin_rescale(da, db, dk, key_mid, out, mid)
        got = out.download()
        # the NTT-form trio of the oracle through the relinearizations
        trios = np.stack([orc.ntt(np.stack([x[0], x[0], x[1]]), mid)
                          for x in a])
        dt = ctx.to_device(trios)
        rel = ctx.array((count, 2, limbs, n))
        ctx.relinearize(dt, dk, key_mid, rel, mid)
        relin = rel.download()
        if log_n == 16 and alpha == 4:
            each = [ctx.to_device(t) for t in trios]
            outs = [ctx.array((2, limbs, n)) for _ in each]
            ctx.relinearize_uneven(each, [mid] * count, dk, key_mid, outs)
            for c in range(count):
                assert np.array_equal(outs[c].download(), relin[c]), c
            for arr in each + outs:
                arr.free()
        for arr in (da, db, dk, out, dt, rel):
            arr.free()
    for c in range(count):
        assert np.array_equal(got[c], orc.hmult(a[c], b[c], key, mid,
                                                key_mid)), c
        assert np.array_equal(relin[c], orc.relinearize(trios[c], key, mid,
                                                        key_mid)), c
