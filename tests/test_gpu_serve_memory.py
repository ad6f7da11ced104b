"""Admission by free memory: the estimate of a batch's working set covers
what its first run takes.  A reserve that leaves exactly that much (measured
on a context of its own) defers the same batch on a fresh context."""
import pytest
import torch

import fhe_amd
from test_gpu_serve import Served

pytestmark = pytest.mark.gpu


def take(log_n, kind, level, count, reserve_of):
    """(device bytes the batch's first run took, deferred admissions)."""
    s = Served(log_n, 7)
    try:
        ctx = s.ctx
        jobs = (fhe_amd.Job * count)()
        for j in range(count):
            a, b = s.duo(level), s.duo(level)
            out = ctx.array(a.shape)
            s.arrays.append(out)
            jobs[j].engine, jobs[j].kind, jobs[j].level = 0, kind, level
            jobs[j].a, jobs[j].b = a.ptr.value, b.ptr.value
            jobs[j].out = out.ptr.value
            jobs[j].arrival_ms = 0.0
        ctx.synchronize()
        free = torch.cuda.mem_get_info()[0]
        stats = fhe_amd.serve([s.engine()], jobs, max_batch=count,
                              reserve_bytes=reserve_of(free))
        ctx.synchronize()
        return free - torch.cuda.mem_get_info()[0], stats.deferred_admissions
    finally:
        s.close()


@pytest.mark.parametrize("log_n,level,count,kind", [
    (15, 10, 2, "dot"), (15, 10, 16, "poly"), (16, 12, 8, "poly")])
def test_estimate_covers_the_first_run(gpu_lib, log_n, level, count, kind):
    code = fhe_amd.JOB_DOT if kind == "dot" else fhe_amd.JOB_POLY
    took, deferred = take(log_n, code, level, count, lambda free: 0)
    assert deferred == 0
    print(f"N=2^{log_n} {kind}: first run took {took >> 20} MiB", flush=True)
    # room for half of it: deferred; for exactly it: deferred too, since the
    # estimate is no smaller
    for share in (0.5, 1.0):
        _, deferred = take(log_n, code, level, count,
                           lambda free: free - int(share * took))
        assert deferred >= 1, (share, took)
    # room for eight times as much: admitted at once
    _, deferred = take(log_n, code, level, count,
                       lambda free: free - 8 * took)
    assert deferred == 0
