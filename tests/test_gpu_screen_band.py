"""The screened index search around its scan: the group-minimum samples of small and middling batches,
the choice of the scan's row tile, and the kernel that turns candidate lists into rerank lists (lists in
LDS, lists too long for it), each against the fp32-only scan of the same live rows bit for bit, with
the handles an index returns after deletions and compaction."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import COSINE, DOT, L2, L2SQ
from tests.test_gpu_index_screen16 import _Index, _fp32_scan

pytestmark = pytest.mark.gpu


def _same(got, want, live):
    gi, gd = got
    wi, wd = want
    none = np.uint32(0xFFFFFFFF)
    np.testing.assert_array_equal(gi, np.where(wi == none, none, live[np.where(wi == none, 0, wi)]))
    np.testing.assert_array_equal(gd.view(np.uint32), wd.view(np.uint32))


def _remove(ctx, ix, rows, compact):
    h = np.ascontiguousarray(rows, dtype=np.uint32)
    ctx.check(ctx.lib.va_index_remove(ctx.handle, ix.h, h.ctypes.data, len(h), None), "va_index_remove")
    if compact:
        ctx.check(ctx.lib.va_index_compact(ctx.handle, ix.h), "va_index_compact")


# 16 | 17 and 32 | 33: the sample's and the scan's tiles; 128 | 129: the scan's; 256 | 257: the sample's;
# 400,000 rows: with deletions the sample's k-th bound is the threshold;
# 98,305 rows: one row past 384 tiles of 256 rows (257 of 384), where the shorter tile is taken
@pytest.mark.parametrize("N,D,Q,k,metric", [(16800, 36, 1, 10, L2SQ), (16801, 64, 16, 3, COSINE), (20001, 100, 17, 10, DOT),
                                            (20001, 128, 32, 10, L2), (16900, 8, 33, 10, COSINE), (98_305, 64, 128, 10, L2SQ),
                                            (98_304, 32, 100, 100, DOT), (30_011, 260, 129, 20, COSINE),
                                            (30_011, 64, 256, 10, L2), (17_001, 64, 257, 10, L2SQ), (400_000, 32, 32, 100, L2SQ)])
@pytest.mark.parametrize("gone", ["none", "masked", "compacted"])
def test_batches(ctx, N, D, Q, k, metric, gone):
    rng = np.random.default_rng(N + Q)
    x = rng.standard_normal((N, D)).astype(np.float32)
    q = rng.standard_normal((Q, D)).astype(np.float32)
    live = np.arange(N, dtype=np.uint32)
    ix = _Index(ctx, x)
    try:
        if gone != "none":
            rows = rng.choice(N, N // 50, replace=False)
            _remove(ctx, ix, rows, gone == "compacted")
            live = np.delete(live, rows)
        gi, gd, t = ix.search(metric, q, k)
        assert t["screened"] == 2 and (gone != "masked" or t["overflow_rows"] == 0), t
        _same((gi, gd), _fp32_scan(ctx, metric, q, x[live], k), live)
    finally:
        ix.close()


@pytest.mark.parametrize("Q", [3, 700])
@pytest.mark.parametrize("rank_of_k,gone", [(True, True), (True, False), (False, False)])
def test_long_lists(ctx, Q, rank_of_k, gone):
    """A 256-row sample and its k-th bound as the threshold: lists of about k N / 256 = 23,000
    candidates, far past the LDS copy; without it (a checked threshold) ordinary ones."""
    from vectoraccelerate_amd import _lib

    N, D, k = 60_000, 32, 100
    rng = np.random.default_rng(Q)
    x = rng.standard_normal((N, D)).astype(np.float32)
    q = rng.standard_normal((Q, D)).astype(np.float32)
    live = np.arange(N, dtype=np.uint32)
    ix = _Index(ctx, x)
    options = {_lib.VA_OPT_SAMPLE_ROWS: 256, _lib.VA_OPT_CANDIDATE_CAP: 32_768}
    if rank_of_k:
        options[_lib.VA_OPT_SAMPLE_RANK] = 2**32
    try:
        if gone:
            rows = rng.choice(N, 500, replace=False)
            _remove(ctx, ix, rows, False)
            live = np.delete(live, rows)
        for o, v in options.items():
            ctx.set_option(o, v)
        gi, gd, t = ix.search(L2SQ, q, k)
        for o in options:
            ctx.set_option(o, 0)
        assert t["screened"] == 2 and (not rank_of_k or t["overflow_rows"] == 0), t
        _same((gi, gd), _fp32_scan(ctx, L2SQ, q, x[live], k), live)
    finally:
        for o in options:
            ctx.set_option(o, 0)
        ix.close()


@pytest.mark.parametrize("Q,k,gone,sample", [(40, 200, True, 4096), (40, 400, True, 16_384), (256, 1000, True, 16_384),
                                             (40, 1000, False, 4096), (32, 1000, True, 4096)])
def test_sample_of_middling_batches(ctx, Q, k, gone, sample):
    """With deletions the lists hold about k N / S rows: middling batches keep the larger sample where
    those would be long."""
    N, D = 60_000, 32
    rng = np.random.default_rng(Q + k)
    x = rng.standard_normal((N, D)).astype(np.float32)
    q = rng.standard_normal((Q, D)).astype(np.float32)
    live = np.arange(N, dtype=np.uint32)
    ix = _Index(ctx, x)
    try:
        if gone:
            rows = rng.choice(N, N // 50, replace=False)
            _remove(ctx, ix, rows, False)
            live = np.delete(live, rows)
        gi, gd, t = ix.search(L2SQ, q, k)
        assert t["screened"] == 2 and t["sample_rows"] == sample, t
        _same((gi, gd), _fp32_scan(ctx, L2SQ, q, x[live], k), live)
    finally:
        ix.close()
