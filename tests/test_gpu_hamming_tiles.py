"""The Hamming filter scan over its resident-query sizes (32, 64, 128, 256) and row widths, with partial
last tiles: exact against the oracle.  A forced sample size keeps the searches on the filter scan."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import check_topk_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 4, 8, 12, 16, 20, 24, 32])
@pytest.mark.parametrize("Q,N,k", [(1, 1025, 3), (32, 3001, 20), (33, 2049, 7), (64, 1056, 64), (65, 4127, 10), (128, 2300, 1),
                                   (129, 2815, 33), (300, 1999, 12)])
def test_filter_scan_tiles(ctx, oracle, W, Q, N, k):
    import torch

    from vectoraccelerate_amd import _lib

    g = np.random.default_rng(W * 1000 + Q)
    x = g.integers(0, 2**32, (N, W), dtype=np.uint64).astype(np.uint32)
    q = g.integers(0, 2**32, (Q, W), dtype=np.uint64).astype(np.uint32)
    x[5], x[N - 1], x[7] = q[Q - 1], 0xFFFFFFFF, 0  # a zero distance, the widest and the narrowest row
    q[0] = 0xFFFFFFFF
    xd, qd = ctx.buffer(x.view(np.int32)), ctx.buffer(q.view(np.int32))
    i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)
    ctx.order_after_torch()
    ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 500)
    try:
        ctx.check(ctx.lib.va_hamming_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, W, k, i.data_ptr(), d.data_ptr()),
                  "va_hamming_topk")
        ctx.synchronize()
    finally:
        ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 0)
    check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy().view(np.uint32), *oracle.hamming_topk(q, x, k))
