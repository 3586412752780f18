// va_select.hip — exact row-wise top-k on 32-bit ordering keys.
//
// One workgroup per row (or per segment of a long dense row):
//   1. radix select (LDS histograms of 11 bits, below the bits all keys share) finds T, the k-th
//      smallest key;
//   2. when more items share T than are needed, a second radix select over the ids of the
//      key == T items finds the cut id, so ties go to the lower index;
//   3. the exactly-k winners are gathered into LDS and bitonic-sorted by (key, id).
// The (distance, index) order is the reference's tie rule (Metal4Common.h:142-159,
// SearchAndRetrieval.metal:313-317); unlike topk_select_batch_kernel
// (SearchAndRetrieval.metal:88-156, value-only compares) the result is deterministic.
#include <algorithm>

#include "va_internal.hpp"
#include "va_select.hpp"

namespace va {
namespace {

// One workgroup per row.  Not CACHED (long rows, lists of a large capacity): a list that turns out
// to hold at most kSelList keys is still copied to LDS.
constexpr uint32_t kSelList = 4096;
template <int NT, bool CACHED, bool KTH = false>
__global__ __launch_bounds__(NT) void select_kernel(SelectArgs a) {
    extern __shared__ uint32_t s_row[];  // the row's keys
    __shared__ SelectLds<KTH> lds;
    const uint32_t row = blockIdx.x;
    if (a.zero_cnt && threadIdx.x == 0) a.zero_cnt[row] = 0;
    if (a.zero_words && row == 0 && threadIdx.x < kZeroWords) a.zero_words[threadIdx.x] = 0;
    if (CACHED || (a.counts && a.counts[row] <= kSelList))
        select_row<NT, true, KTH>(a, row, lds, s_row);
    else
        select_row<NT, false, KTH>(a, row, lds, s_row);
    if constexpr (KTH)
        if (a.ptc && threadIdx.x == 0) {  // (the thread that wrote the threshold)
            const float4 inf = a.qinfo[row];
            const PreTest p = pretest_consts(a.bound, inf.x, inf.y, inf.z, inf.w, a.out_kth[row]);
            a.ptc[row] = float4{p.A, p.B, p.C, inf.z};
        }
}

// float values -> ordering keys (dense matrices given to va_topk_select)
__global__ void keys_from_floats(const float* v, uint64_t n, int desc, uint32_t* out) {
    uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const uint64_t step = uint64_t(gridDim.x) * blockDim.x;
    for (; i < n; i += step) out[i] = desc ? key_of_float_desc(v[i]) : key_of_float(v[i]);
}

// two sorted k-lists per row -> 2k candidate (key, id) pairs; sentinels dropped
__global__ void merge_gather(const uint32_t* ai, const float* ad, const uint32_t* bi, const float* bd, uint32_t rows,
                             uint32_t k, uint32_t chunk_base, uint32_t* ckey, uint32_t* cid, uint32_t* ccnt) {
    const uint32_t row = blockIdx.x;
    __shared__ uint32_t s_n;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < 2 * k; r += blockDim.x) {
        const bool from_a = r < k;
        const uint32_t j = from_a ? r : r - k;
        const uint32_t id = from_a ? ai[int64_t(row) * k + j] : bi[int64_t(row) * k + j];
        if (id == kSentinel) continue;
        const float d = from_a ? ad[int64_t(row) * k + j] : bd[int64_t(row) * k + j];
        const uint32_t p = atomicAdd(&s_n, 1u);
        ckey[int64_t(row) * 2 * k + p] = key_of_float(d);
        cid[int64_t(row) * 2 * k + p] = from_a ? id : id + chunk_base;
    }
    __syncthreads();
    if (threadIdx.x == 0) ccnt[row] = s_n;
}

}  // namespace

va_status launch_select(va_context* ctx, const SelectArgs& a) {
    if (a.rows == 0) return VA_OK;
    if (a.k > SEL_BUF) return fail(ctx, VA_ERR_INVALID_ARG, "k=%u exceeds the maximum %u", a.k, SEL_BUF);
    // Candidate lists are mostly far below their capacity, which sizes the LDS copy: past 8K
    // entries a large copy would leave one workgroup per CU, so such rows are read from memory
    // (L2-resident lists) by many workgroups at once instead; and so are dense rows of that length
    // when not all of them would be on the chip at once (1,000 rows of 16,384 keys, k = 600
    // 321 -> 118 us; 600 of 8,193, which are, 70 from their copies, 78 without).
    const uint32_t n = a.nseg ? a.seg : a.n;
    constexpr uint32_t kLds = 160 * 1024;
    const bool resident = a.rows <= uint64_t(ctx->num_cus) * (kLds / (n * 4ull + sizeof(SelectLds<false>)));
    const bool cache = n <= 8192 || (n <= kSelCache && !a.counts && !a.out_kth && resident);
    const size_t lds = size_t(cache ? std::max<uint32_t>(n, 1) : (a.counts ? kSelList : 0)) * 4;
    auto go = [&](auto kern, int threads) -> va_status {
        if (lds > 48 * 1024)
            VA_CHECK_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        kern<<<dim3(a.rows), dim3(threads), lds, ctx->stream>>>(a);
        return VA_OK;
    };
    // A few long rows: 1,024 threads each, since a row's passes are a serial chain and the chip has
    // room; many rows share a CU with 256.
    const bool tall = n > 1024 && a.rows <= 2 * uint32_t(ctx->num_cus);
    if (a.out_kth)
        VA_CHECK_STATUS(cache ? (tall ? go(&select_kernel<1024, true, true>, 1024) : go(&select_kernel<256, true, true>, 256))
                              : (tall ? go(&select_kernel<1024, false, true>, 1024)
                                      : go(&select_kernel<256, false, true>, 256)));
    else
        VA_CHECK_STATUS(cache ? (tall ? go(&select_kernel<1024, true>, 1024) : go(&select_kernel<256, true>, 256))
                              : (tall ? go(&select_kernel<1024, false>, 1024) : go(&select_kernel<256, false>, 256)));
    VA_CHECK_LAUNCH(ctx);
    return VA_OK;
}

va_status launch_select_dense(va_context* ctx, const SelectArgs& a, const SegmentPlan& seg, uint32_t* wkey,
                              uint32_t* wid) {
    if (seg.n <= 1) return launch_select(ctx, a);
    SelectArgs p;
    p.keys = a.keys;
    p.ld = a.ld;
    p.n = a.n;
    p.rows = a.rows * seg.n;
    p.k = a.k;
    p.seg = seg.len;
    p.nseg = seg.n;
    p.key_bits = a.key_bits;
    p.spread = a.spread;
    p.out_idx = wid;
    p.out_key = wkey;
    VA_CHECK_STATUS(launch_select(ctx, p));
    SelectArgs m = a;
    m.keys = wkey;
    m.ids = wid;
    m.ld = int64_t(seg.n) * a.k;
    m.n = seg.n * a.k;
    m.spread = false;
    return launch_select(ctx, m);
}

}  // namespace va

extern "C" {

va_status va_topk_select(va_context* ctx, const float* values, uint32_t num_rows, uint32_t num_elements, uint32_t k,
                         va_select_mode mode, uint32_t* out_idx, float* out_values) {
    if (!ctx) return VA_ERR_INVALID_ARG;
    VA_REQUIRE(ctx, values && out_idx, "va_topk_select: NULL pointer");
    VA_REQUIRE(ctx, num_rows > 0 && num_elements > 0, "va_topk_select: empty input");
    VA_REQUIRE(ctx, k > 0 && k <= VA_MAX_K, "va_topk_select: k must be in [1, %u], got %u", VA_MAX_K, k);
    VA_REQUIRE(ctx, mode == VA_SELECT_MIN || mode == VA_SELECT_MAX, "va_topk_select: bad mode");
    va::DeviceGuard g(ctx->device);
    const uint64_t total = uint64_t(num_rows) * num_elements;
    va::Scratch s(ctx);
    const va::SegmentPlan seg = va::select_segments(num_elements, k, num_rows, uint32_t(ctx->num_cus));
    const uint64_t win = uint64_t(num_rows) * seg.n * k;
    VA_CHECK_STATUS(s.reserve(va::Scratch::round(total * 4) + va::Scratch::round(win * 4) * 2));
    uint32_t* keys = s.carve<uint32_t>(total);
    uint32_t* wkey = s.carve<uint32_t>(win);
    uint32_t* wid = s.carve<uint32_t>(win);
    uint64_t blocks = (total + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    va::keys_from_floats<<<dim3(uint32_t(blocks)), dim3(256), 0, ctx->stream>>>(values, total, mode == VA_SELECT_MAX,
                                                                                keys);
    VA_CHECK_LAUNCH(ctx);
    va::SelectArgs a;
    a.keys = keys;
    a.ld = num_elements;
    a.n = num_elements;
    a.rows = num_rows;
    a.k = k;
    a.out_idx = out_idx;
    a.out_f = out_values;
    a.key_kind = mode == VA_SELECT_MAX ? 1 : 0;
    a.spread = true;
    return va::launch_select_dense(ctx, a, seg, wkey, wid);
}

va_status va_topk_merge(va_context* ctx, const uint32_t* a_idx, const float* a_dist, const uint32_t* b_idx,
                        const float* b_dist, uint32_t num_rows, uint32_t k, uint32_t chunk_base, uint32_t* out_idx,
                        float* out_dist) {
    if (!ctx) return VA_ERR_INVALID_ARG;
    VA_REQUIRE(ctx, a_idx && a_dist && b_idx && b_dist && out_idx, "va_topk_merge: NULL pointer");
    VA_REQUIRE(ctx, num_rows > 0, "va_topk_merge: empty input");
    VA_REQUIRE(ctx, k > 0 && k <= VA_MAX_K, "va_topk_merge: k must be in [1, %u], got %u", VA_MAX_K, k);
    va::DeviceGuard g(ctx->device);
    const uint64_t cand = uint64_t(num_rows) * 2 * k;
    va::Scratch s(ctx);
    VA_CHECK_STATUS(s.reserve(va::Scratch::round(cand * 4) * 2 + va::Scratch::round(uint64_t(num_rows) * 4)));
    uint32_t* ckey = s.carve<uint32_t>(cand);
    uint32_t* cid = s.carve<uint32_t>(cand);
    uint32_t* ccnt = s.carve<uint32_t>(num_rows);
    va::merge_gather<<<dim3(num_rows), dim3(256), 0, ctx->stream>>>(a_idx, a_dist, b_idx, b_dist, num_rows, k,
                                                                     chunk_base, ckey, cid, ccnt);
    VA_CHECK_LAUNCH(ctx);
    va::SelectArgs a;
    a.keys = ckey;
    a.ids = cid;
    a.counts = ccnt;
    a.ld = 2 * k;
    a.n = 2 * k;
    a.rows = num_rows;
    a.k = k;
    a.out_idx = out_idx;
    a.out_f = out_dist;
    return va::launch_select(ctx, a);
}

}  // extern "C"
