"""The Hamming filter scan over its resident-query sizes (32, 64, 128, 256) and row widths, with partial
last tiles: exact against the oracle.  A forced sample size keeps the searches on the filter scan."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import check_topk_exact

pytestmark = pytest.mark.gpu


def _search(ctx, oracle, x, q, k):
    """Exact, over a sample of 500 rows: the filter scan."""
    import torch

    from vectoraccelerate_amd import _lib

    (N, W), Q = x.shape, len(q)
    xd, qd = ctx.buffer(x.view(np.int32)), ctx.buffer(q.view(np.int32))
    i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)
    ctx.order_after_torch()
    ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 500)
    ctx.set_profiling(True)
    try:
        ctx.check(ctx.lib.va_hamming_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, W, k, i.data_ptr(), d.data_ptr()),
                  "va_hamming_topk")
        t = ctx.last_scan_timings()
    finally:
        ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 0)
        ctx.set_profiling(False)
    assert t["sample_rows"] == 500, t  # the filter scan ran (dense keys take no sample)
    check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy().view(np.uint32), *oracle.hamming_topk(q, x, k))


@pytest.mark.parametrize("W", [1, 4, 8, 12, 16, 20, 24, 32])
@pytest.mark.parametrize("Q,N,k", [(1, 1025, 3), (32, 3001, 20), (33, 2049, 7), (64, 1056, 64), (65, 4127, 10), (128, 2300, 1),
                                   (129, 2815, 33), (300, 1999, 12)])
def test_filter_scan_tiles(ctx, oracle, W, Q, N, k):
    g = np.random.default_rng(W * 1000 + Q)
    x = g.integers(0, 2**32, (N, W), dtype=np.uint64).astype(np.uint32)
    q = g.integers(0, 2**32, (Q, W), dtype=np.uint64).astype(np.uint32)
    x[5], x[N - 1], x[7] = q[Q - 1], 0xFFFFFFFF, 0  # a zero distance, the widest and the narrowest row
    q[0] = 0xFFFFFFFF
    _search(ctx, oracle, x, q, k)


@pytest.mark.parametrize("W", [4, 24, 32])
@pytest.mark.parametrize("Q", [25, 32, 64, 100, 128, 200])
@pytest.mark.parametrize("kind", ["runs", "all"])
def test_staged_passes(ctx, oracle, W, Q, kind):
    """Equal queries, and rows equal to them: a wave appends all 64 passes of two rows at once, onto
    stages that hold any number already.  "runs": runs of 1 to 64 such rows among others; "all": every
    row, so every list overflows and the fallback finds the top-k."""
    g = np.random.default_rng(W * 1000 + Q)
    N = 6000
    q = np.tile(g.integers(0, 2**32, (1, W), dtype=np.uint64).astype(np.uint32), (Q, 1))
    x = g.integers(0, 2**32, (N, W), dtype=np.uint64).astype(np.uint32)
    if kind == "all":
        x[:] = q[0]
    for r in range(100, N - 64, 300):
        x[r : r + 1 + r // 9 % 64] = q[0]
    _search(ctx, oracle, x, q, 20)
