"""Workspaces of key switching below N = 2^16, which holds every partition of
a group of ciphertexts: where they may not grow (a captured graph holds their
addresses) calls whose one-partition form fits run in smaller groups or that
form; products with a key need no more than relinearizing them; a large
batch's extended limbs stay bounded; results may overlap the factors of the
allocation-free product.  Each against the same call with room."""
import ctypes

import numpy as np
import pytest
import torch

import fhe_amd
from test_gpu_small_rings import uniform

pytestmark = pytest.mark.gpu


def fixed(ctx, words):
    """A context whose scratch holds about `words` words from now on (a
    product without a key takes 2 x 2 x limbs x N of it per ciphertext), with
    a graph alive.  Returns the graph."""
    level = 1
    limbs = ctx.limbs_at(ctx.info["full_level"] - level)
    out_limbs = limbs - 1
    count = words // (4 * limbs * ctx.n)
    a = ctx.to_device(np.zeros((count, 2, limbs, ctx.n), np.int64))
    out = ctx.array((count, 3, out_limbs, ctx.n))
    ctx.multiply(a, level, 0, a, level, 0, out)
    ctx.synchronize()
    ctx.graph_begin()
    ctx.multiply(a, level, 0, a, level, 0, out)
    graph = ctx.graph_end()
    a.free()
    out.free()
    return graph


# room in limbs per ciphertext beside the start of the buffer: the
# one-partition form only, groups of one, and all but a few limbs of the batch
@pytest.mark.parametrize("log_n,alpha,limbs", [(13, 1, 3), (14, 1, 8),
                                               (15, 2, 7)])
@pytest.mark.parametrize("form", ["one partition", "groups of one",
                                  "groups of two"])
def test_fixed_workspace(gpu_lib, log_n, alpha, limbs, form):
    count = 3
    got = []
    for limited in (False, True):
        with fhe_amd.Context(log_n, alpha) as ctx:
            rng = np.random.Generator(np.random.PCG64(40))
            n, key_mid = ctx.n, ctx.key_moduli_id()
            mid = ctx.chain_count - limbs
            ext = limbs + alpha
            parts = -(-limbs // alpha)
            trios = uniform(rng, ctx.primes, mid, (count, 3, limbs, n))
            key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
            graph = None
            if limited:
                others = count * (3 * limbs + 2 * ext)
                extra = {"one partition": count * ext,
                         "groups of one": parts * ext,
                         "groups of two": 2 * parts * ext}[form]
                low = ctx.limbs_at(ctx.info["full_level"] - 1)
                graph = fixed(ctx, (others + extra + 4 * low) * n)
            dt, dk = ctx.to_device(trios), ctx.to_device(key)
            duos = ctx.to_device(np.ascontiguousarray(trios[:, :2]))
            rel, sw, rot, conj = (ctx.array((count, 2, limbs, n))
                                  for _ in range(4))
            outs = [ctx.array((count, 2, limbs, n)) for _ in range(2)]
            print(f"fixed workspace N=2^{log_n} {form}", flush=True)
            ctx.relinearize(dt, dk, key_mid, rel, mid)
            ctx.switch_key(duos, dk, key_mid, sw, mid)
            ctx.rotate(duos, dk, key_mid, 3, rot, mid)
            ctx.conjugate(duos, dk, key_mid, conj, mid)
            ctx.rotate_batch(duos, [dk, dk], [key_mid] * 2, [1, 2], outs, mid)
            got.append([x.download() for x in [rel, sw, rot, conj] + outs])
            if graph is not None:
                ctx.graph_destroy(graph)
            for arr in [dt, dk, duos, rel, sw, rot, conj] + outs:
                arr.free()
    assert [np.array_equal(x, y) for x, y in zip(*got)] == [True] * 6


@pytest.mark.parametrize("log_n,alpha", [(14, 1), (16, 4)])
def test_product_needs_no_more_than_relinearizing(gpu_lib, log_n, alpha):
    count, level = 2, 4
    with fhe_amd.Context(log_n, alpha) as ctx:
        rng = np.random.Generator(np.random.PCG64(41))
        n, key_mid = ctx.n, ctx.key_moduli_id()
        mid = ctx.info["full_level"] - level
        limbs, out_limbs = ctx.limbs_at(mid), ctx.limbs_at(mid) - 1
        key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
        a = uniform(rng, ctx.primes, mid, (2 * count, 2, limbs, n))
        dk, both = ctx.to_device(key), ctx.to_device(a)
        x, y = ctx.to_device(a[:count]), ctx.to_device(a[count:])
        trio = ctx.array((2 * count, 3, out_limbs, n))
        want = ctx.array((count, 2, out_limbs, n))
        got = ctx.array((count, 2, out_limbs, n))
        half = ctx.array((count, 3, out_limbs, n))
        # the stash as large as a product of twice the texts makes it, the
        # scratch as large as the relinearization asks for
        ctx.multiply(both, level, 0, both, level, 0, trio)
        ctx.multiply(x, level, 0, y, level, 0, half)
        ctx.relinearize(half, dk, key_mid, want, mid + 1)
        ctx.synchronize()
        ctx.graph_begin()
        ctx.relinearize(half, dk, key_mid, want, mid + 1)
        graph = ctx.graph_end()
        ctx.multiply(x, level, 0, y, level, 0, got, dk, key_mid)
        same = np.array_equal(got.download(), want.download())
        ctx.graph_destroy(graph)
        for arr in (dk, both, x, y, trio, want, got, half):
            arr.free()
    assert same


def test_large_batch_is_bounded(gpu_lib):
    """400 key switches at N = 2^15 with 18 limbs: 21 GB of extended limbs
    and digits at once, in groups of at most 8 GiB."""
    count, limbs, alpha = 400, 18, 2
    with fhe_amd.Context(15, alpha) as ctx:
        rng = np.random.Generator(np.random.PCG64(42))
        n, key_mid = ctx.n, ctx.key_moduli_id()
        mid = ctx.chain_count - limbs
        one = uniform(rng, ctx.primes, mid, (2, limbs, n))
        key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
        dk, single = ctx.to_device(key), ctx.to_device(one[None])
        want = ctx.array((1, 2, limbs, n))
        ctx.switch_key(single, dk, key_mid, want, mid)
        many = ctx.array((count, 2, limbs, n))
        out = ctx.array((count, 2, limbs, n))
        for c in range(count):
            many.upload_at(one, c * one.size)
        ctx.synchronize()
        before = torch.cuda.mem_get_info()[0]
        print("large batch", flush=True)
        ctx.switch_key(many, dk, key_mid, out, mid)
        ctx.synchronize()
        grown = before - torch.cuda.mem_get_info()[0]
        expect = want.download()[0]
        host = np.empty_like(expect)
        same = []
        for c in range(0, count, 7):
            fhe_amd._check(fhe_amd.library().fhe_copy_to_host(
                ctx.handle, host.ctypes.data,
                ctypes.c_void_p(out.ptr.value + c * host.nbytes),
                host.nbytes))
            same.append(np.array_equal(host, expect))
        for arr in (dk, single, want, many, out):
            arr.free()
    assert all(same)
    accumulators = count * 2 * (limbs + alpha) * n * 8
    assert grown < accumulators + (9 << 30), grown


def test_noalloc_result_over_factors(gpu_lib):
    """Results written over the factors, from the second pair on: a batch
    that runs in parts must have read a factor before its place is taken."""
    with fhe_amd.Context(15, 2) as ctx:
        n, limbs, count = ctx.n, 18, 7
        mid, key_mid = ctx.chain_count - limbs, ctx.key_moduli_id()
        rng = np.random.Generator(np.random.PCG64(43))
        a = uniform(rng, ctx.primes, mid, (count, 2, limbs, n))
        key = uniform(rng, ctx.primes, key_mid, ctx.key_shape(key_mid), 2)
        # room for the results from the second pair's place on
        da, dk = ctx.array((count + 1, 2, limbs, n)), ctx.to_device(key)
        factors = ctx.to_device(a)
        want = ctx.array((count, 2, limbs - 1, n))
        ctx.hmult_relin_rescale(factors, factors, dk, key_mid, want, mid)
        expect = want.download()
        same = []
        for start in (0, 1):
            da.upload_at(a, 0)
            at = ctypes.c_void_p(da.ptr.value + start * a[0].nbytes)
            assert fhe_amd.library().fhe_hmult_relin_rescale_noalloc(
                ctx.handle, count, mid, da.ptr, da.ptr, dk.ptr, key_mid,
                at) == 0
            got = da.download().reshape(-1)[start * a[0].size:]
            same.append(np.array_equal(got[:expect.size],
                                       expect.reshape(-1)))
        for arr in (da, dk, factors, want):
            arr.free()
    assert same == [True, True]
