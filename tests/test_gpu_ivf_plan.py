"""The inverted-list search's plan at the edges of its one-launch form (probes, pairs, lists), of its one
workgroup (with lists that end within the last of several) and of the
tile groups that a batch can need, long lists shared out among the waves of the 16-query tiles (their
stages overflow), with the probes a caller may pass (repeated, out of range): against
the oracle, and the screened scan against the fp32 list scan bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import L2SQ, check_topk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,D,N,Q,nprobe,k", [(1, 36, 500, 3, 1, 10), (16, 64, 3000, 16, 4, 10), (16, 64, 3000, 17, 4, 10),
                                              (40, 32, 4000, 32, 8, 5), (40, 32, 4000, 33, 8, 5), (64, 32, 6000, 64, 64, 10),
                                              (65, 32, 6000, 63, 65, 10), (64, 32, 6000, 65, 64, 3),
                                              (8192, 16, 20_000, 5, 20, 10), (8193, 16, 20_000, 5, 20, 10),
                                              (2048, 16, 20_000, 70, 65, 10), (2049, 16, 20_000, 70, 65, 10),
                                              (20_001, 16, 60_000, 70, 8, 10), (20_001, 9, 60_000, 500, 9, 10),
                                              (30, 768, 3000, 128, 2, 10), (30, 768, 3000, 129, 2, 10), (5, 33, 700, 9, 3, 10),
                                              (3, 64, 30_000, 4, 2, 100), (2, 128, 70_001, 16, 2, 1)])
@pytest.mark.parametrize("odd_probes", [False, True])
def test_plan(ctx, oracle, C, D, N, Q, nprobe, k, odd_probes):
    import torch

    from vectoraccelerate_amd import IVFSearchConfiguration, IVFSearchPipeline, _lib

    g = np.random.default_rng(C + Q)
    x = g.standard_normal((N, D)).astype(np.float32)
    q = g.standard_normal((Q, D)).astype(np.float32)
    pipe = IVFSearchPipeline(ctx, IVFSearchConfiguration(C, nprobe, D))
    st = pipe.prepareIndexStructure(x[g.choice(N, C, replace=False)], x)
    probes = pipe.findNearestCentroids(q, st).cpu().numpy().view(np.uint32).copy()
    if odd_probes:
        probes[::2, -1] = probes[::2, 0]  # repeated
        probes[1::3, 0] = 0xFFFFFFFF      # missing
        probes[2::5, -1] = C              # out of range
    pd, qd = ctx.buffer(probes.view(np.int32)), ctx.buffer(q)
    outs = []
    for screen in (0, 1):
        i, d = ctx.empty((Q, k), torch.int32), ctx.empty((Q, k), torch.float32)
        ctx.order_after_torch()
        ctx.set_option(_lib.VA_OPT_SCREEN, screen)
        try:
            ctx.check(ctx.lib.va_ivf_scan(ctx.handle, st.handle, qd.data_ptr(), Q, pd.data_ptr(), nprobe, k, i.data_ptr(),
                                          d.data_ptr()), "va_ivf_scan")
            ctx.synchronize()
        finally:
            ctx.set_option(_lib.VA_OPT_SCREEN, 0)
        outs.append((i.cpu().numpy().view(np.uint32), d.cpu().numpy()))
    np.testing.assert_array_equal(outs[0][0], outs[1][0])
    np.testing.assert_array_equal(outs[0][1].view(np.uint32), outs[1][1].view(np.uint32))
    off, ids = st.lists()
    once = probes.copy()  # a list is scanned once however often it is named
    for row in once:
        row[[j for j in range(nprobe) if row[j] in row[:j]]] = 0xFFFFFFFF
    oi, od = oracle.ivf_scan(q, x, off, ids, once, k)
    check_topk(L2SQ, q, x, k, *outs[0], oi, od)
    st.close()
