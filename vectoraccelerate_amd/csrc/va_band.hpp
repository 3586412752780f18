// va_band.hpp — from a screened query's candidates to its rerank list in one kernel (the flat
// screen and the IVF list scan): the interval of every pair, the k-th smallest upper bound u, and
// the candidates whose lower bound is within u (every row of the top-k is among them).
//
// The three steps as kernels of their own (intervals, selection, compaction) cost a launch each and
// passed the intervals through memory twice; here they stay in LDS.  One workgroup per query;
// lists past band_list entries keep their intervals in place in memory.
#pragma once

#include <algorithm>

#include "va_select.hpp"

namespace va {

// Intervals kept in LDS, and the launch of a band kernel kern<NT>: 8,192 entries leave room for two
// workgroups of 1,024 threads per CU, 4,096 for four of 512 (few queries take 1,024 threads each, as
// the selections do).
constexpr uint32_t kBandList = 8192;
inline bool band_tall(const va_context* ctx, uint32_t Q) { return Q <= 2 * uint32_t(ctx->num_cus); }
inline uint32_t band_list(bool tall, uint32_t cap) {
    return std::min<uint32_t>(tall ? kBandList : kBandList / 2, (cap + 63) / 64 * 64);
}

struct BandArgs {
    const uint32_t* cnt = nullptr;  // [Q] candidates appended (may exceed cap: the list overflowed)
    uint32_t* hi = nullptr;         // [Q x cap] in: the unscaled fp16 dot; scratch for long lists
    uint32_t* lo = nullptr;         // [Q x cap] in (flat): |x|^2; scratch for long lists
    const uint32_t* id = nullptr;   // [Q x cap] candidates
    uint32_t cap = 0, k = 0, min_count = 0;
    uint32_t list = 0;  // band_list(cap)
    // u beyond thr[q] lists the query for the fallback (fewer than k candidates have their upper
    // bound within the threshold the list was filtered with, so it may miss a row); nullptr: no check
    const uint32_t* thr = nullptr;
    // candidates excluded (skip[id], or skip[skip_id[id]]) never count
    const uint8_t* skip = nullptr;
    const uint32_t* skip_id = nullptr;
    // threshold mode: u is written to out_kth[q] and there is no rerank list
    uint32_t* out_kth = nullptr;
    uint32_t* rr = nullptr;      // [Q x rcap]
    uint32_t* rcount = nullptr;  // [Q]
    uint32_t rcap = 0;
    // queries whose list overflowed, fell short of min_count or outgrows rcap: listed for the exact
    // fallback, rcount 0
    uint32_t* ovf_cnt = nullptr;
    uint32_t* ovf_rows = nullptr;
};

struct BandLds : RadixLds {
    uint32_t n;
};

// Every thread of the NT-thread workgroup calls it.  bounds(o, klo, khi): the keys of the interval of
// candidate o (its index in the [Q x cap] arrays).  s: 2 x a.list words of LDS.
template <int NT, class Bounds>
__device__ inline void band_row(const BandArgs& a, uint32_t q, BandLds& lds, uint32_t* s, Bounds&& bounds) {
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t n = a.cnt[q];
    auto give_up = [&] {
        if (tid == 0 && a.ovf_cnt) {
            a.rcount[q] = 0;
            a.ovf_rows[atomicAdd(a.ovf_cnt, 1u)] = q;
        }
        if (tid == 0 && a.out_kth) a.out_kth[q] = 0xFFFFFFFFu;
    };
    if (n > a.cap || n < a.min_count) return give_up();
    const int64_t o = int64_t(q) * a.cap;
    auto run = [&](uint32_t* hi, uint32_t* lo) {
        uint32_t mn = 0xFFFFFFFFu, mx = 0;
        // (four pairs per thread in flight: their rows' norms are gathered through the ids)
        for (uint32_t i0 = tid; i0 < n; i0 += 4 * NT) {
            uint32_t klo[4], khi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) bounds(o + min(i0 + uint32_t(j) * NT, n - 1), klo[j], khi[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t i = i0 + uint32_t(j) * NT;
                if (i >= n) break;
                if (a.skip) {
                    const uint32_t id = a.id[o + i];
                    if (a.skip[a.skip_id ? a.skip_id[id] : id]) klo[j] = khi[j] = kAbsentKey;
                }
                hi[i] = khi[j];
                lo[i] = klo[j];
                mn = min(mn, khi[j]);
                mx = max(mx, khi[j]);
            }
        }
        if (tid == 0) lds.n = 0;
        __syncthreads();
        uint32_t u = 0xFFFFFFFFu;
        if (n > a.k) {
            uint32_t need = a.k, eq = n;
            u = kth_key<NT>(
                lds,
                [&](auto&& f) {
                    for (uint32_t i = tid; i < n; i += NT) f(hi[i]);
                },
                mn, mx, need, eq);
        }
        if (a.out_kth) {
            if (tid == 0) a.out_kth[q] = u;
            return;
        }
        if (a.thr && u > a.thr[q]) return give_up();
        uint32_t* out = a.rr + int64_t(q) * a.rcap;
        for (uint32_t i0 = 0; i0 < n; i0 += NT) {
            const uint32_t i = i0 + uint32_t(tid);
            const uint32_t l = i < n ? lo[i] : kAbsentKey;
            const bool p = l <= u && l != kAbsentKey;
            const uint64_t b = __ballot(p);
            uint32_t base = 0;
            if (lane == 0 && b) base = atomicAdd(&lds.n, uint32_t(__popcll(b)));
            base = __shfl(base, 0);
            if (p) {
                const uint32_t pos = base + uint32_t(__popcll(b & ((1ull << lane) - 1)));
                if (pos < a.rcap) out[pos] = a.id[o + i];
            }
        }
        __syncthreads();
        const uint32_t m = lds.n;
        if (m > a.rcap) return give_up();
        if (tid == 0) a.rcount[q] = m;
    };
    if (n <= a.list) run(s, s + a.list);
    else run(a.hi + o, a.lo + o);
}

}  // namespace va
