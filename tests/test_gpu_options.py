"""Every pipeline choice of fhe_context_set_option gives the same limbs: the
batched Gold-size HMult+relin+rescale under each option equals the default
pipeline's output bit for bit (the default is itself checked against the
reference digests and the oracle in test_gpu_hmult.py), and so does the key
product split over blocks (one ciphertext) against the unsplit one (the same
ciphertext in a batch)."""
import numpy as np
import pytest

import fhe_amd
from support import golden, hmult_inputs
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu

DEFAULTS = {"own_limbs": 1, "staged_modup": 1, "ks_lazy_accumulate": 1,
            "lazy_key_switch": 1}
OPTIONS = [{"own_limbs": 0}, {"staged_modup": 0}, {"ks_lazy_accumulate": 0},
           {"lazy_key_switch": 0}, {"staged_modup": 0, "own_limbs": 0},
           {"staged_modup": 0, "lazy_key_switch": 0},
           {"own_limbs": 0, "lazy_key_switch": 0}]
# names of pipelines that the defaults have replaced
RETIRED = {"split_variants": 0, "overlap_trio": 2, "ks_wide_accumulate": 1,
           "ks_prefetch": 1, "ks_occupancy": 3, "fuse_tensor": 1,
           "fuse_modup": 1}


def test_options_bit_identical(gpu_lib):
    case = [c for c in golden("hmult_golden.json")["cases"]
            if c["name"] == "gold_mid30"][0]
    n = 1 << case["log_n"]
    limbs = case["limbs"]
    A, B, K = hmult_inputs(case["primes"], n, case["moduli_id"], limbs,
                           case["key_moduli_id"], case["key_polys"],
                           case["key_chain"], case["seed"])
    with fhe_amd.Context(case["log_n"], case["special_prime_count"],
                         primes=case["primes"]) as ctx:
        count = 3
        da = ctx.to_device(np.stack([A] * count))
        db = ctx.to_device(np.stack([B] * count))
        dk = ctx.to_device(K.reshape(case["key_polys"], case["key_chain"], n))
        out = ctx.array((count, 2, limbs - 1, n))

        def run():
            ctx.hmult_relin_rescale(da, db, dk, case["key_moduli_id"], out,
                                    case["moduli_id"])
            return out.download()

        want = run()
        for opts in OPTIONS:
            print(f"options {opts}", flush=True)
            for name, value in opts.items():
                ctx.set_option(name, value)
            got = run()
            for name in opts:
                ctx.set_option(name, DEFAULTS[name])
            assert np.array_equal(got, want), opts
        for name, value in RETIRED.items():
            ctx.set_option(name, value)
        assert np.array_equal(run(), want)
        with pytest.raises(fhe_amd.FheError):
            ctx.set_option("no_such_option", 1)
        for arr in (da, db, dk, out):
            arr.free()


@pytest.mark.parametrize("log_n,alpha,limbs", [(13, 1, 3), (14, 1, 8),
                                               (14, 3, 5), (15, 8, 9),
                                               (16, 4, 3)])
def test_small_rings_and_batches(gpu_lib, log_n, alpha, limbs):
    """The options on one ciphertext, whose key product is split over blocks
    (partition groups, and key halves on the smallest), and on a batch, whose
    key product is not."""
    count = 64 if log_n < 15 else 16
    with fhe_amd.Context(log_n, alpha) as ctx:
        rng = np.random.Generator(np.random.PCG64(50))
        n, mid, key_mid = ctx.n, ctx.chain_count - limbs, ctx.key_moduli_id()
        one = uniform(rng, ctx.primes, mid, (1, 2, limbs, n))
        key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
        dk, single = ctx.to_device(key), ctx.to_device(one)
        many = ctx.to_device(np.repeat(one, count, 0))
        out1 = ctx.array((1, 2, limbs - 1, n))
        outs = ctx.array((count, 2, limbs - 1, n))
        want = None
        for opts in [{}] + OPTIONS:
            print(f"N=2^{log_n} options {opts}", flush=True)
            for name, value in opts.items():
                ctx.set_option(name, value)
            ctx.hmult_relin_rescale(single, single, dk, key_mid, out1, mid)
            ctx.hmult_relin_rescale(many, many, dk, key_mid, outs, mid)
            for name in opts:
                ctx.set_option(name, DEFAULTS[name])
            got, batch = out1.download(), outs.download()
            want = got if want is None else want
            assert np.array_equal(got, want), opts
            same = all(np.array_equal(b, want[0]) for b in batch)
            assert same, opts
        for arr in (dk, single, many, out1, outs):
            arr.free()
