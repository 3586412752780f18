"""Dense keys and their selection: rows cut into segments, the histogram passes with ties and crowded
bins, the streamed fp32 kernel at the edges of its tiles and chunks (bit for bit the distance GEMM's
values), and the sampled scans of small batches that the dense path otherwise replaces."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import COSINE, DOT, L2, L2SQ, check_topk, check_topk_exact

pytestmark = pytest.mark.gpu


def _select(ctx, v, k, mode):
    import torch

    rows, n = v.shape
    dv = ctx.buffer(v)
    i, o = ctx.empty((rows, k), torch.int32), ctx.empty((rows, k), torch.float32)
    ctx.order_after_torch()
    ctx.check(ctx.lib.va_topk_select(ctx.handle, dv.data_ptr(), rows, n, k, mode, i.data_ptr(), o.data_ptr()), "select")
    ctx.synchronize()
    return i.cpu().numpy().view(np.uint32), o.cpu().numpy()


@pytest.mark.parametrize("rows,n,k", [(1, 8192, 10), (1, 8193, 10), (3, 12289, 1), (2, 100_003, 100), (1, 65_537, 1024),
                                      (600, 9000, 7), (5, 1500, 129), (4, 128, 128), (2, 40, 60),
                                      # the lowest id among the ties of the smallest key; rows read from
                                      # memory, cut (k = 32) and whole (more of them than half the CUs)
                                      (3, 100, 1), (140, 26_000, 1), (140, 26_000, 32), (140, 26_000, 33),
                                      (140, 9000, 33), (400, 17_000, 300)])
@pytest.mark.parametrize("kind", ["spread", "ties", "crowded"])
@pytest.mark.parametrize("mode", [0, 1])
def test_select_rows(ctx, oracle, rows, n, k, kind, mode):
    """Values are copied, never computed: exact.  Ties cross the segments (lower index first);
    "crowded" puts all values but a few within one part in 1e6, with NaN, infinities and -0."""
    g = np.random.default_rng(n + k)
    if kind == "spread":
        v = g.standard_normal((rows, n)).astype(np.float32)
    elif kind == "ties":
        v = g.integers(-3, 4, (rows, n)).astype(np.float32)
    else:
        v = (1000.0 + 1e-3 * g.random((rows, n))).astype(np.float32)
        v[:, :: max(1, n // 9)] *= -1.0
        v[:, 3] = np.nan
        v[:, 5] = np.inf
        v[:, 7] = -np.inf
        v[:, 11] = -0.0
        v[:, 13] = 0.0
    gi, gv = _select(ctx, v, k, mode)
    oi, ov = oracle.topk_rows(v, k, mode_max=bool(mode))
    np.testing.assert_array_equal(gi, oi)
    kk = min(k, n)
    np.testing.assert_array_equal(np.where(gv[:, :kk] == 0, 0, gv[:, :kk]), np.where(ov[:, :kk] == 0, 0, ov[:, :kk]))


@pytest.mark.parametrize("rows,n,k", [(1, 16_789_505, 10), (2, 20_480_001, 10), (1, 20_480_001, 1024)])
def test_select_rows_of_many_segments(ctx, oracle, rows, n, k):
    """Rows past 4096^2 values, where the segments' length rounds up enough that one fewer covers the
    row.  The winners lie at both ends, and the rows differ there: values read from beyond a row, or
    winners counted twice, would be among the results."""
    g = np.random.default_rng(n)
    v = np.tile(g.random((1, 1 << 20), dtype=np.float32), (rows, n // (1 << 20) + 1))[:, :n].copy()
    half = min(k, 40) // 2
    for r in range(rows):
        v[r, :half] = -1.0 - 3.0 * r - np.arange(half, dtype=np.float32) / 64
        v[r, n - half:] = -2.0 - 3.0 * r - np.arange(half, dtype=np.float32) / 64
    gi, gv = _select(ctx, v, k, 0)
    oi, ov = oracle.topk_rows(v, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gv, ov)


@pytest.mark.parametrize("metric", [L2SQ, COSINE, DOT, L2])
@pytest.mark.parametrize("Q,N,D", [(1, 1, 1), (1, 31, 3), (2, 32, 15), (31, 33, 16), (32, 95, 17), (33, 127, 32), (5, 129, 36),
                                   (40, 200, 48), (3, 97, 100), (65, 64, 127), (1, 300, 128), (17, 161, 130), (100, 250, 260)])
def test_streamed_keys_equal_the_gemm(ctx, metric, Q, N, D):
    """k = N: the search's distances are every key of the streamed kernel, and equal the all-pairs
    GEMM's values bit for bit (its queries take another kernel)."""
    import torch

    g = np.random.default_rng(Q + N + D + metric)
    q, x = ctx.buffer(g.standard_normal((Q, D), dtype=np.float32)), ctx.buffer(g.standard_normal((N, D), dtype=np.float32))
    i, d = ctx.empty((Q, N), torch.int32), ctx.empty((Q, N), torch.float32)
    m = ctx.empty((Q, N), torch.float32)
    ctx.order_after_torch()
    ctx.check(ctx.lib.va_fused_topk(ctx.handle, metric, q.data_ptr(), x.data_ptr(), Q, N, D, N, i.data_ptr(), d.data_ptr()),
              "va_fused_topk")
    if metric == DOT:
        ctx.check(ctx.lib.va_dot_all_pairs(ctx.handle, q.data_ptr(), x.data_ptr(), m.data_ptr(), Q, N, D, 0), "dot")
    elif metric == COSINE:
        ctx.check(ctx.lib.va_cosine_all_pairs(ctx.handle, q.data_ptr(), x.data_ptr(), m.data_ptr(), Q, N, D, 1), "cosine")
    else:
        ctx.check(ctx.lib.va_l2_all_pairs(ctx.handle, q.data_ptr(), x.data_ptr(), m.data_ptr(), Q, N, D, int(metric == L2)),
                  "l2")
    ctx.synchronize()
    if metric == DOT:
        m = -m
    ids = i.long()
    assert bool((ids.sort(dim=1).values == torch.arange(N, device=ids.device)).all())
    got = torch.empty_like(d).scatter_(1, ids, d)
    np.testing.assert_array_equal((got + 0.0).cpu().numpy().view(np.uint32), (m + 0.0).cpu().numpy().view(np.uint32))


@pytest.mark.parametrize("Q,k", [(1, 1), (7, 10), (33, 40), (90, 100), (180, 5)])
def test_sampled_scans_of_small_batches(ctx, oracle, Q, k):
    """A forced sample size sends batches that would take the dense path through the sampled scan:
    threshold from group minima (k = 1, 10, 5) and from the sample itself, filter, selection."""
    import torch

    from vectoraccelerate_amd import _lib

    g = np.random.default_rng(Q + k)
    N, D = 12_345, 64
    x, q = g.standard_normal((N, D), dtype=np.float32), g.standard_normal((Q, D), dtype=np.float32)
    xc, qc = g.integers(-128, 128, (N, D)).astype(np.int8), g.integers(-128, 128, (Q, D)).astype(np.int8)
    xb = g.integers(0, 2**32, (N, 8), dtype=np.uint64).astype(np.uint32)
    qb = g.integers(0, 2**32, (Q, 8), dtype=np.uint64).astype(np.uint32)
    L, p = ctx.lib, lambda t: t.data_ptr()  # noqa: E731
    dev = [ctx.buffer(a) for a in (x, q, xc, qc, xb.view(np.int32), qb.view(np.int32))]
    out = [(ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.float32 if j == 0 else torch.int32)) for j in range(3)]
    ctx.order_after_torch()
    ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 2048)
    try:
        ctx.check(L.va_fused_topk(ctx.handle, L2SQ, p(dev[1]), p(dev[0]), Q, N, D, k, p(out[0][0]), p(out[0][1])), "fused")
        ctx.check(L.va_i8_scan_topk(ctx.handle, p(dev[3]), p(dev[2]), Q, N, D, k, p(out[1][0]), p(out[1][1])), "i8")
        ctx.check(L.va_hamming_topk(ctx.handle, p(dev[5]), p(dev[4]), Q, N, 8, k, p(out[2][0]), p(out[2][1])), "hamming")
        ctx.synchronize()
    finally:
        ctx.set_option(_lib.VA_OPT_SAMPLE_ROWS, 0)
    host = [(i.cpu().numpy().view(np.uint32), d.cpu().numpy()) for i, d in out]
    check_topk(L2SQ, q, x, k, *host[0], *oracle.flat_topk(L2SQ, q, x, k))
    check_topk_exact(*host[1], *oracle.i8_topk(qc, xc, k))
    check_topk_exact(host[2][0], host[2][1].view(np.uint32), *oracle.hamming_topk(qb, xb, k))


@pytest.mark.parametrize("Q,N,D", [(40, 74_678, 2048), (40, 74_679, 2048), (9, 1_000_000, 1732), (9, 1_000_000, 1736)])
def test_filter_streamed_or_gemm(ctx, Q, N, D):
    """Either side of the line between the streamed filter pass and the GEMM's, at Q past and below 32: the
    same keys, those of the all-pairs GEMM bit for bit (ties to the lower id)."""
    import torch

    k = 20
    gen = torch.Generator(device="cuda").manual_seed(N)
    x, q = torch.randn(N, D, device="cuda", generator=gen), torch.randn(Q, D, device="cuda", generator=gen)
    i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.float32)
    m = ctx.empty((Q, N), torch.float32)
    ctx.order_after_torch()
    ctx.check(ctx.lib.va_fused_topk(ctx.handle, L2SQ, q.data_ptr(), x.data_ptr(), Q, N, D, k, i.data_ptr(), d.data_ptr()),
              "va_fused_topk")
    ctx.check(ctx.lib.va_l2_all_pairs(ctx.handle, q.data_ptr(), x.data_ptr(), m.data_ptr(), Q, N, D, 0), "l2")
    ctx.synchronize()
    want, ids = m.sort(dim=1, stable=True)
    np.testing.assert_array_equal(d.cpu().numpy(), want[:, :k].cpu().numpy())
    np.testing.assert_array_equal(i.cpu().numpy(), ids[:, :k].to(torch.int32).cpu().numpy())


@pytest.mark.parametrize("N,Q,k,dense", [(400_003, 1, 10, True), (400_003, 1, 300, False), (400_003, 4, 600, True),
                                         (900_001, 4, 300, False)])
def test_dense_or_sampled(ctx, oracle, N, Q, k, dense):
    """Either side of the line in the winners that one workgroup would merge per row: exact."""
    import torch

    g = np.random.default_rng(N + k)
    x = g.integers(0, 2**32, (N, 2), dtype=np.uint64).astype(np.uint32)
    q = g.integers(0, 2**32, (Q, 2), dtype=np.uint64).astype(np.uint32)
    xd, qd = ctx.buffer(x.view(np.int32)), ctx.buffer(q.view(np.int32))
    i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.int32)
    ctx.order_after_torch()
    ctx.set_profiling(True)
    try:
        ctx.check(ctx.lib.va_hamming_topk(ctx.handle, qd.data_ptr(), xd.data_ptr(), Q, N, 2, k, i.data_ptr(), d.data_ptr()),
                  "va_hamming_topk")
        t = ctx.last_scan_timings()
    finally:
        ctx.set_profiling(False)
    assert (t["sample_rows"] == 0) == dense, t
    check_topk_exact(i.cpu().numpy().view(np.uint32), d.cpu().numpy().view(np.uint32), *oracle.hamming_topk(q, x, k))
