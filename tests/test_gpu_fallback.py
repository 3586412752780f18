"""The one-launch overflow fallback (va_fallback.hpp): every phase of it over the slot counts where
its work items change (32 queries per group, 64 queries per grid size), on searches queued back to
back so that each finds its phase words cleared, against the unforced search bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import check_topk_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,N,D,k", [(1, 3001, 20, 1), (31, 5000, 33, 12), (33, 2500, 64, 100), (64, 4099, 16, 7),
                                     (65, 4099, 16, 7), (130, 2049, 8, 300)])
def test_every_query_overflows(ctx, oracle, Q, N, D, k):
    """int8 codes of a narrow range (heavy ties: a query's tie list overflows for some shapes), a
    64-entry candidate list, rank k: every query with more than 64 candidates takes the fallback.
    Three searches queued without a synchronisation must each give the oracle's result."""
    import torch

    from vectoraccelerate_amd import _lib

    rng = np.random.default_rng(Q + N)
    x = rng.integers(-2, 3, (N, D)).astype(np.int8)
    q = rng.integers(-2, 3, (Q, D)).astype(np.int8)
    xd, qd = ctx.buffer(x), ctx.buffer(q)
    outs = [(ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)) for _ in range(3)]
    ctx.order_after_torch()
    for option, value in ((_lib.VA_OPT_CANDIDATE_CAP, 64), (_lib.VA_OPT_SAMPLE_ROWS, 512), (_lib.VA_OPT_SAMPLE_RANK, 2**32)):
        ctx.set_option(option, value)
    ctx.set_profiling(True)
    try:
        for i, d in outs:
            ctx.check(ctx.lib.va_i8_scan_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, D, k, i.data_ptr(),
                                              d.data_ptr()), "va_i8_scan_topk")
        ctx.synchronize()
        t = ctx.last_scan_timings()
    finally:
        ctx.set_profiling(False)
        for option in (_lib.VA_OPT_CANDIDATE_CAP, _lib.VA_OPT_SAMPLE_ROWS, _lib.VA_OPT_SAMPLE_RANK):
            ctx.set_option(option, 0)
    if k > 1:
        assert t["overflow_rows"] > 0, t
    oi, od = oracle.i8_topk(q, x, k)
    for i, d in outs:
        check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy(), oi, od)


@pytest.mark.parametrize("N,W", [(2500, 2), (40_000, 4)])
@pytest.mark.parametrize("Q,listed", [(66, [0]), (300, [3, 299]), (300, list(range(0, 300, 7)))])
def test_few_of_many_queries_overflow(ctx, oracle, N, W, Q, listed):
    """A launch of the full grid for a few listed queries: fewer slots than workgroups, and (N = 2500) fewer
    work items.  Only the listed queries have more rows at one distance than their candidate list holds."""
    import torch

    from vectoraccelerate_amd import _lib

    k = 5
    g = np.random.default_rng(N + Q)
    x = g.integers(0, 2**32, (N, W), dtype=np.uint64).astype(np.uint32)
    q = g.integers(0, 2**32, (Q, W), dtype=np.uint64).astype(np.uint32)
    q[listed] = x[7]
    x[200:1700] = x[7]
    xd, qd = ctx.buffer(x.view(np.int32)), ctx.buffer(q.view(np.int32))
    outs = [(ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)) for _ in range(2)]
    ctx.order_after_torch()
    for option, value in ((_lib.VA_OPT_CANDIDATE_CAP, 1400), (_lib.VA_OPT_SAMPLE_ROWS, 1000)):
        ctx.set_option(option, value)
    ctx.set_profiling(True)
    try:
        for i, d in outs:
            ctx.check(ctx.lib.va_hamming_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, W, k, i.data_ptr(),
                                              d.data_ptr()), "va_hamming_topk")
        ctx.synchronize()
        t = ctx.last_scan_timings()
    finally:
        ctx.set_profiling(False)
        for option in (_lib.VA_OPT_CANDIDATE_CAP, _lib.VA_OPT_SAMPLE_ROWS):
            ctx.set_option(option, 0)
    assert len(listed) <= t["overflow_rows"] < Q, t
    oi, od = oracle.hamming_topk(q, x, k)
    for i, d in outs:
        check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy().view(np.uint32), oi, od)
