// va_scan.hip — exact top-k scan driver shared by the fp32, int8 and binary search paths.
//
// The reference picks between a fused K<=8 shader and a two-pass path that materialises
// the Q x N distance matrix in 64 MB chunks (FusedL2TopKKernel.execute,
// Kernels/Metal4/FusedL2TopKKernel.swift:367-427, :765-1090).  Here every k takes one path
// and the full matrix is never stored:
//   1. sample:  dense keys of each query against S strided rows; tau_q = the r-th smallest
//               (r = k: an upper bound of the true k-th key, since the sample rows are real
//               rows and the filter pass computes bit-identical keys for them; r < k: a
//               tighter threshold that is checked in step 3, see sample_rank);
//   2. filter:  the scan kernel appends every key <= tau_q to the query's candidate list;
//   3. select:  exact (key, id) top-k of every candidate list that holds at least k keys
//               (then every key of the top-k is <= tau_q, so all of them are in the list);
//   4. overflow: rows whose list outgrew its capacity, or fell short of k, are recomputed
//               exactly by chunked dense keys + select + a final select over the per-chunk
//               winners.
#include <algorithm>
#include <cmath>
#include <vector>

#include "va_fallback.hpp"
#include "va_internal.hpp"

namespace va {

__global__ void mask_dense_kernel(uint32_t* keys, uint32_t cols, int64_t ld, uint32_t row0, uint32_t stride,
                                  const uint8_t* __restrict__ skip) {
    uint32_t* k = keys + int64_t(blockIdx.y) * ld;
    for (uint32_t j = blockIdx.x * 256 + threadIdx.x; j < cols; j += gridDim.x * 256)
        if (skip[row0 + uint64_t(j) * stride]) k[j] = kAbsentKey;
}

__global__ void mask_list_kernel(uint32_t* keys, const uint32_t* __restrict__ ids,
                                 const uint32_t* __restrict__ counts, uint32_t cap, int64_t ld,
                                 const uint8_t* __restrict__ skip) {
    const uint32_t r = blockIdx.y;
    const uint32_t n = min(counts[r], cap);
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const int64_t o = int64_t(r) * ld + i;
        const uint32_t id = ids[o];
        if (id != kSentinel && skip[id]) keys[o] = kAbsentKey;
    }
}

va_status mask_dense_keys(va_context* ctx, uint32_t* keys, uint32_t rows, uint32_t cols, int64_t ld, uint32_t row0,
                          uint32_t stride, const uint8_t* skip) {
    if (!skip || rows == 0 || cols == 0) return VA_OK;
    const uint32_t bx = std::min<uint32_t>(64, (cols + 255) / 256);
    for (uint32_t r0 = 0; r0 < rows; r0 += 65535) {
        const uint32_t nr = std::min<uint32_t>(65535, rows - r0);
        mask_dense_kernel<<<dim3(bx, nr), dim3(256), 0, ctx->stream>>>(keys + int64_t(r0) * ld, cols, ld, row0, stride,
                                                                      skip);
        VA_CHECK_LAUNCH(ctx);
    }
    return VA_OK;
}

va_status mask_list_keys(va_context* ctx, uint32_t* keys, const uint32_t* ids, const uint32_t* counts, uint32_t rows,
                         uint32_t cap, int64_t ld, const uint8_t* skip) {
    if (!skip || rows == 0 || cap == 0) return VA_OK;
    const uint32_t bx = std::min<uint32_t>(16, (cap + 255) / 256);
    for (uint32_t r0 = 0; r0 < rows; r0 += 65535) {
        const uint32_t nr = std::min<uint32_t>(65535, rows - r0);
        mask_list_kernel<<<dim3(bx, nr), dim3(256), 0, ctx->stream>>>(keys + int64_t(r0) * ld, ids + int64_t(r0) * ld,
                                                                     counts + r0, cap, ld, skip);
        VA_CHECK_LAUNCH(ctx);
    }
    return VA_OK;
}

// gmin[r * G + g] = the smallest of the keys r * ld + g + j G, j < kGroupKeys (columns past S
// absent).  Any partition of the sample into groups will do; this one reads whole lines.
constexpr uint32_t kGroupKeys = 32;
__global__ __launch_bounds__(256) void group_min_kernel(const uint32_t* __restrict__ keys, int64_t ld, uint32_t S,
                                                        uint32_t G, uint32_t* __restrict__ gmin) {
    const uint32_t g = blockIdx.x * 256 + threadIdx.x;
    if (g >= G) return;
    const uint32_t* row = keys + int64_t(blockIdx.y) * ld;
    uint32_t v[kGroupKeys];
#pragma unroll
    for (uint32_t j = 0; j < kGroupKeys; ++j) v[j] = g + j * G < S ? row[g + j * G] : 0xFFFFFFFFu;
    uint32_t m = v[0];
#pragma unroll
    for (uint32_t j = 1; j < kGroupKeys; ++j) m = min(m, v[j]);
    gmin[int64_t(blockIdx.y) * G + g] = m;
}

bool fb_fits(const va_context* ctx, size_t need, uint32_t rows, uint32_t N, uint32_t k) {
    return fb_fits_in(ctx->fixed_scratch ? ctx->fixed_scratch_bytes : 0, need, rows, N, k);
}

size_t dense_budget(const va_context* ctx) {
    return dense_budget_for(ctx->fixed_scratch ? ctx->fixed_scratch_bytes : 0);
}

// (The screened scan took N/32 sample rows while its threshold was the sample's k-th bound; with
// the checked smaller rank N/64 is faster there too: configs[1] 3.98 -> 3.84 ms per search.)
ScanPlan plan_scan(const va_context* ctx, uint32_t Q, uint32_t N, uint32_t k) {
    return plan_scan_for(dense_budget(ctx), ctx->opt_sample_rows, ctx->opt_candidate_cap, Q, N, k);
}

va_status rescan_rows(va_context* ctx, KeyProducer& kp, uint32_t N, uint32_t k, const SelectArgs& base,
                      const uint32_t* rows_dev, uint32_t n_rows, const uint8_t* skip) {
    if (n_rows == 0) return VA_OK;
    // The row list is read back first: the arena below may be regrown (which frees it).
    std::vector<uint32_t> rows_host(n_rows);
    VA_CHECK_HIP(ctx, hipMemcpyAsync(rows_host.data(), rows_dev, size_t(n_rows) * 4, hipMemcpyDeviceToHost,
                                     ctx->stream));
    VA_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    // rows are processed in batches of R; each batch scans the database in chunks of C rows
    // (a fixed scratch block halves R until the batch fits)
    const uint64_t budget = dense_budget(ctx);
    uint32_t R = std::min<uint32_t>(n_rows, 64), C = 0, nch = 0;
    size_t need = 0;
    for (;;) {
        C = uint32_t(std::max<uint64_t>(k, std::min<uint64_t>(N, budget / (uint64_t(R) * 4))));
        nch = (N + C - 1) / C;
        need = Scratch::round(uint64_t(n_rows) * 4) + Scratch::round(uint64_t(R) * C * 4) +
               Scratch::round(uint64_t(R) * nch * k * 4) * 2;
        if (!ctx->fixed_scratch || need <= ctx->fixed_scratch_bytes || R == 1) break;
        R = (R + 1) / 2;
    }
    Scratch f(ctx);
    VA_CHECK_STATUS(f.reserve(need));
    uint32_t* ovf_rows = f.carve<uint32_t>(n_rows);
    uint32_t* dkeys = f.carve<uint32_t>(uint64_t(R) * C);
    uint32_t* wkey = f.carve<uint32_t>(uint64_t(R) * nch * k);
    uint32_t* wid = f.carve<uint32_t>(uint64_t(R) * nch * k);
    VA_CHECK_HIP(ctx, hipMemcpyAsync(ovf_rows, rows_host.data(), size_t(n_rows) * 4, hipMemcpyHostToDevice,
                                     ctx->stream));
    for (uint32_t r0 = 0; r0 < n_rows; r0 += R) {
        const uint32_t nr = std::min(R, n_rows - r0);
        const uint32_t* rows = ovf_rows + r0;
        for (uint32_t c = 0; c < nch; ++c) {
            const uint32_t c0 = c * C;
            const uint32_t cols = std::min(C, N - c0);
            VA_CHECK_STATUS(kp.dense(rows, 0, nr, c0, cols, 1, dkeys, C));
            VA_CHECK_STATUS(mask_dense_keys(ctx, dkeys, nr, cols, C, c0, 1, skip));
            SelectArgs a;
            a.keys = dkeys;
            a.ld = C;
            a.n = cols;
            a.rows = nr;
            a.k = k;
            a.id_offset = c0;
            a.out_ld = int64_t(nch) * k;
            a.out_idx = wid + int64_t(c) * k;
            a.out_key = wkey + int64_t(c) * k;
            VA_CHECK_STATUS(launch_select(ctx, a));
        }
        SelectArgs a = base;
        a.keys = wkey;
        a.ids = wid;
        a.counts = nullptr;
        a.ld = int64_t(nch) * k;
        a.n = nch * k;
        a.rows = nr;
        a.row_map = rows;
        a.overflow_count = nullptr;
        a.overflow_rows = nullptr;
        VA_CHECK_STATUS(launch_select(ctx, a));
    }
    // the host copy of the row list must outlive the upload above
    VA_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return VA_OK;
}

// The order statistic of the sample that becomes a query's threshold (sample_rank_for): with
// r < k the filter keeps about r N / S rows instead of k N / S, and a query is short of k
// candidates exactly when r of its k nearest rows are in the sample (then the select lists it for
// the exact fallback).
uint32_t sample_rank(const va_context* ctx, uint32_t k, uint64_t S, uint32_t N, bool masked) {
    return sample_rank_for(ctx->opt_sample_rank, k, S, N, masked);
}

// Up to this many (query, row) pairs a search writes every key and selects from them: two or three
// launches instead of the sampled scan's five or six and its second pass over part of the rows.
// Measured per search, k = 10, dense against sampled: fp32 768-d, 50,000 rows, Q = 8 57 / 83 us,
// Q = 40 (2M pairs) 107 / 129, 200,000 rows, Q = 40 (8M) 290 / 286; int8 512-d, 20,000 rows, Q = 160
// (3.2M) 53 / 56, 50,000 rows, Q = 160 (8M) 89 / 68; PQ, 500,000 rows, Q = 8 (4M) 80 / 83.
// One workgroup merges the winners of a long row's segments, about n k / max(4096, 16 k) of them, which
// for a large k takes longer than a sample and a filter pass; those take longer with Q k.  us, dense /
// sampled (one board): Hamming 256-bit, Q = 1, 300,000 rows, k = 100 40 / 41, 300 63 / 52; 3.9M rows, k = 100
// 124 / 62, 500 261 / 83; Q = 4, 600,000 rows, k = 300 93 / 74, 1000 101 / 116; int8 64-d, 900,000 rows, Q = 1,
// k = 200 71 / 54; Q = 4, k = 1000 104 / 115; fp32 64-d, 3.9M rows, Q = 1, k = 10 290 / 298, 200 393 / 306.
constexpr uint64_t kDensePairs = 4ull << 20;
static bool dense_pays(const va_context* ctx, uint32_t Q, uint32_t N, uint32_t k) {
    const uint64_t winners = uint64_t(select_segments(N, k, Q, uint32_t(ctx->num_cus)).n) * k;
    return uint64_t(Q) * N <= kDensePairs && winners <= 10240 + 16ull * Q * k;
}
va_status exact_topk_scan(va_context* ctx, KeyProducer& kp, uint32_t Q, uint32_t N, uint32_t k,
                          const ScanOutputs& out) {
    SelectArgs base;
    base.k = k;
    base.out_idx = out.idx;
    base.out_map = out.map;
    base.out_f = out.f;
    base.out_i32 = out.i32;
    base.out_key = out.key;
    base.key_kind = out.key_kind;
    base.key_bits = kp.key_bits();

    // ---- plan ------------------------------------------------------------------------
    const bool automatic = !ctx->opt_candidate_cap && !ctx->opt_sample_rows && !ctx->opt_sample_rank;
    const ScanPlan plan = plan_scan(ctx, Q, N, k);
    const uint64_t S = plan.S;
    const bool direct =
        plan.direct || (automatic && dense_pays(ctx, Q, N, k) && uint64_t(Q) * N * 4 <= dense_budget(ctx));
    ScanPhaseMarks pm(ctx);
    ctx->last_scan = va_scan_timings{};
    VA_CHECK_STATUS(pm.mark(0));
    if (direct) {
        ctx->last_scan.scan_launches = 0;
        // small database: dense keys in query chunks + select
        const uint64_t per_q = uint64_t(N) * 4;
        uint32_t qc = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(Q, dense_budget(ctx) / per_q)));
        const SegmentPlan seg = select_segments(N, k, qc, uint32_t(ctx->num_cus));
        const uint64_t win = uint64_t(qc) * seg.n * k;  // winners of the rows' segments
        Scratch s(ctx);
        VA_CHECK_STATUS(s.reserve(Scratch::round(uint64_t(qc) * per_q) + Scratch::round(win * 4) * 2));
        uint32_t* keys = s.carve<uint32_t>(uint64_t(qc) * N);
        uint32_t* wkey = s.carve<uint32_t>(win);
        uint32_t* wid = s.carve<uint32_t>(win);
        for (uint32_t q0 = 0; q0 < Q; q0 += qc) {
            const uint32_t nq = std::min(qc, Q - q0);
            VA_CHECK_STATUS(kp.dense(nullptr, q0, nq, 0, N, 1, keys, N));
            VA_CHECK_STATUS(mask_dense_keys(ctx, keys, nq, N, N, 0, 1, out.skip));
            ctx->last_scan.scan_launches++;
            SelectArgs a = base;
            a.keys = keys;
            a.ld = N;
            a.n = N;
            a.rows = nq;
            if (out.idx) a.out_idx = out.idx + int64_t(q0) * k;
            if (out.f) a.out_f = out.f + int64_t(q0) * k;
            if (out.i32) a.out_i32 = out.i32 + int64_t(q0) * k;
            if (out.key) a.out_key = out.key + int64_t(q0) * k;
            VA_CHECK_STATUS(launch_select_dense(ctx, a, seg, wkey, wid));
        }
        return pm.finish(false, false);
    }
    const uint32_t stride = plan.stride;
    const uint64_t cap = plan.cap;
    const uint32_t rank = sample_rank(ctx, k, S, N, out.skip != nullptr);
    const uint32_t qs = plan.qs;
    // The threshold may be looser than the sample's rank-th key (a rank below k is checked by the
    // selection, rank k only needs an upper bound of the k-th key), so it is the rank-th smallest
    // of the minima of groups of keys: one workgroup per query over the whole sample row was a
    // serial pass of 16K-260K keys (10M int8 rows, Q = 32: 263 us on 32 workgroups, now 20).
    // The minima sit where the candidate lists go later.
    const uint32_t groups = ceil_div(S, kGroupKeys);
    const bool group_min = S >= 128ull * rank && uint64_t(qs) * groups <= 2 * uint64_t(Q) * cap;

    Scratch s(ctx);
    size_t need = exact_scan_need(Q, plan);
    // overflowed rows are finished on the device (no read-back) when the fallback's buffers fit
    const bool device_fb = fb_fits(ctx, need, Q, N, k);
    if (device_fb) need += fb_bytes(Q, N, k);
    VA_CHECK_STATUS(s.reserve(need));
    uint32_t* thr = s.carve<uint32_t>(Q);
    uint32_t* cnt = s.carve<uint32_t>(Q);
    uint32_t* ovf_rows = s.carve<uint32_t>(Q);
    uint32_t* ckey = s.carve<uint32_t>(uint64_t(Q) * cap);
    uint32_t* cid = s.carve<uint32_t>(uint64_t(Q) * cap);
    uint32_t* ovf_cnt = s.carve<uint32_t>(kZeroWords);
    uint32_t* skeys = s.carve<uint32_t>(uint64_t(qs) * S);
    uint32_t* const gkeys = ckey;  // (ckey and cid are adjacent)
    FbArgs fb;
    if (device_fb) {
        fb = fb_carve(s, Q, N, k);
        fb.n_rows = ovf_cnt;
        fb.rows = ovf_rows;
        fb.sync = ovf_cnt + kFbSync;
        fb.skip = out.skip;
    }
    VA_CHECK_STATUS(s.verify(need));

    // ---- 1. sample thresholds -----------------------------------------------------------
    for (uint32_t q0 = 0; q0 < Q; q0 += qs) {
        const uint32_t nq = std::min(qs, Q - q0);
        VA_CHECK_STATUS(kp.dense(nullptr, q0, nq, 0, uint32_t(S), stride, skeys, int64_t(S)));
        VA_CHECK_STATUS(mask_dense_keys(ctx, skeys, nq, uint32_t(S), int64_t(S), 0, stride, out.skip));
        if (group_min)
            for (uint32_t r0 = 0; r0 < nq; r0 += 65535) {
                const uint32_t nr = std::min<uint32_t>(65535, nq - r0);
                group_min_kernel<<<dim3((groups + 255) / 256, nr), dim3(256), 0, ctx->stream>>>(
                    skeys + uint64_t(r0) * S, int64_t(S), uint32_t(S), groups, gkeys + uint64_t(r0) * groups);
                VA_CHECK_LAUNCH(ctx);
            }
        SelectArgs a;
        a.keys = group_min ? gkeys : skeys;
        a.n = group_min ? groups : uint32_t(S);
        a.ld = int64_t(a.n);
        a.rows = nq;
        a.k = rank;
        a.out_kth = thr + q0;
        a.key_bits = kp.key_bits();
        a.zero_cnt = cnt + q0;  // the filter's list lengths and overflow words
        a.zero_words = ovf_cnt;
        VA_CHECK_STATUS(launch_select(ctx, a));
    }
    // ---- 2. filter --------------------------------------------------------------------
    VA_CHECK_STATUS(pm.mark(1));
    VA_CHECK_STATUS(kp.filter(thr, cnt, ckey, cid, uint32_t(cap)));
    VA_CHECK_STATUS(pm.mark(2));
    VA_CHECK_STATUS(mask_list_keys(ctx, ckey, cid, cnt, Q, uint32_t(cap), int64_t(cap), out.skip));
    ctx->last_scan.scan_launches = 1;
    ctx->last_scan.sample_rows = uint32_t(S);
    ctx->last_scan.candidate_cap = uint32_t(cap);
    // ---- 3. select ----------------------------------------------------------------------
    {
        SelectArgs a = base;
        a.keys = ckey;
        a.ids = cid;
        a.counts = cnt;
        a.ld = int64_t(cap);
        a.n = uint32_t(cap);
        a.rows = Q;
        a.overflow_count = ovf_cnt;
        a.overflow_rows = ovf_rows;
        a.min_count = rank < k ? k : 0;
        VA_CHECK_STATUS(launch_select(ctx, a));
    }
    if (device_fb) VA_CHECK_STATUS(pm.count_overflow(ovf_cnt));  // profiling only
    VA_CHECK_STATUS(pm.mark(3));
    if (device_fb) {
        // ---- 4. exact top-k of the overflowed rows, on the device ------------------------------
        VA_CHECK_STATUS(kp.fallback(fb, fb_select_args(fb, base, kp.key_bits())));
        return pm.finish(true, true);
    }
    VA_CHECK_HIP(ctx, hipMemcpyAsync(ctx->host_word, ovf_cnt, 4, hipMemcpyDeviceToHost, ctx->stream));
    VA_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const uint32_t n_ovf = ctx->host_word[0];
    ctx->last_scan.overflow_rows = n_ovf;
    if (n_ovf == 0) return pm.finish(true, false);

    // ---- 4. exact chunked recomputation of overflowed rows ---------------------------------
    VA_CHECK_STATUS(rescan_rows(ctx, kp, N, k, base, ovf_rows, n_ovf, out.skip));
    return pm.finish(true, true);
}

}  // namespace va
