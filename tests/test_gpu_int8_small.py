"""The int8 scan of small batches (va_int8_small.hip): row lengths that end inside a load, a k-step or a
chunk, every query-block size and the batches past it, partial last tiles; filter scan and dense keys,
exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import check_topk_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sample", [0, 600])
@pytest.mark.parametrize("D", [4, 16, 20, 60, 64, 100, 128, 132, 200, 256, 260, 384, 512, 516, 768, 772, 1020, 1024, 1028])
@pytest.mark.parametrize("Q,N,k", [(1, 1057, 1), (16, 2001, 10), (17, 1500, 5), (33, 999, 20), (65, 3003, 3), (128, 1281, 12),
                                   (131, 2047, 10), (260, 1100, 4)])
def test_small_scan(ctx, oracle, D, Q, N, k, sample):
    """sample 600: the filter scan; 0: dense keys.  Extreme codes reach the largest dots of both signs."""
    import torch

    from vectoraccelerate_amd import _lib

    g = np.random.default_rng(D * 100 + Q)
    x, q = g.integers(-128, 128, (N, D)).astype(np.int8), g.integers(-128, 128, (Q, D)).astype(np.int8)
    x[3], x[4], x[N - 1], q[0], q[Q - 1] = -128, 127, q[Q - 1], -128, 127
    xd, qd = ctx.buffer(x), ctx.buffer(q)
    i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)
    ctx.order_after_torch()
    ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, sample)
    try:
        ctx.check(ctx.lib.va_i8_scan_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, D, k, i.data_ptr(), d.data_ptr()),
                  "va_i8_scan_topk")
        ctx.synchronize()
    finally:
        ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 0)
    check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy(), *oracle.i8_topk(q, x, k))


@pytest.mark.parametrize("D", [20, 64, 512, 528])
@pytest.mark.parametrize("Q,N", [(32, 500), (33, 2047), (64, 2048), (65, 4095), (128, 4096)])
def test_dense_keys_of_few_rows(ctx, oracle, D, Q, N):
    """Either side of the lines below which the LDS-tiled kernel takes the dense keys."""
    test_small_scan(ctx, oracle, D, Q, N, 7, 0)
