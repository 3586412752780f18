// va_select.hpp — the row selection of va_select.hip as a device function, for kernels that end in
// a selection of their own (the overflow fallback).
#pragma once

#include "va_internal.hpp"

namespace va {

constexpr int SEL_THREADS = 256;
constexpr uint32_t SEL_BUF = VA_MAX_K;  // winners buffer (k <= VA_MAX_K)

// Rows of up to kSelCache keys are first copied into LDS (one pass with many loads in flight);
// the radix passes then read LDS instead of re-reading the row from memory once per pass with
// one load in flight per thread, which left a short row's workgroup waiting on memory latency.
constexpr uint32_t kSelCache = 24576;  // 96 KiB

template <bool CACHED>
struct RowView {
    const uint32_t* keys;  // the row in memory, or its copy in LDS
    const uint32_t* ids;
    uint32_t n;
    __device__ uint32_t key(uint32_t i) const { return keys[i]; }
    __device__ uint32_t id(uint32_t i) const { return ids ? ids[i] : i; }
};

// Wave 0 scans the 256-bin histogram and finds the bin holding the `need`-th item.
// Writes digit, the count before it, and the bin count to shared memory.
__device__ inline void find_digit(const uint32_t* hist, uint32_t need, uint32_t* s_digit, uint32_t* s_before,
                           uint32_t* s_bin) {
    const int lane = threadIdx.x & 63;
    if (threadIdx.x >= 64) return;
    uint32_t c[4];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c[i] = hist[lane * 4 + i];
        sum += c[i];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t o = __shfl_up(incl, off);
        if (lane >= off) incl += o;
    }
    uint32_t excl = incl - sum;
    if (excl < need && need <= incl) {
        uint32_t run = excl;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (run < need && need <= run + c[i]) {
                *s_digit = uint32_t(lane * 4 + i);
                *s_before = run;
                *s_bin = c[i];
            }
            run += c[i];
        }
    }
}

// The bin of a histogram of nb <= 2048 bins holding the need-th item: each thread sums eight
// bins, a block-wide scan of the sums, then the thread whose range holds the item finds it.
__device__ inline void find_bin_wide(const uint32_t* hist, uint32_t nb, uint32_t need, uint32_t* s_digit,
                              uint32_t* s_before, uint32_t* s_bin) {
    __shared__ uint32_t wsum[SEL_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint32_t c[8], sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t b = uint32_t(tid) * 8 + i;
        c[i] = b < nb ? hist[b] : 0u;
        sum += c[i];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t base = 0;
    for (int i = 0; i < w; ++i) base += wsum[i];
    incl += base;
    const uint32_t excl = incl - sum;
    if (excl < need && need <= incl) {
        uint32_t run = excl;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (run < need && need <= run + c[i]) {
                *s_digit = uint32_t(tid) * 8 + i;
                *s_before = run;
                *s_bin = c[i];
            }
            run += c[i];
        }
    }
}

// Adds this lane's item to the histogram when m.  Keys of one search crowd into few digits
// (the top bytes of nearby distances are equal; Hamming distances are below 1024), and 256
// threads incrementing one LDS bin serialise: when every active lane of the wave adds to the
// same bin, one lane adds the wave's count.
__device__ __forceinline__ void hist_add(uint32_t* hist, bool m, uint32_t d) {
    const uint32_t dd = m ? d : 0xFFFFFFFFu;
    const uint32_t first = __builtin_amdgcn_readfirstlane(dd);
    const uint64_t act = __ballot(1);
    if (__ballot(dd == first) == act) {
        if (first != 0xFFFFFFFFu && (threadIdx.x & 63) == uint32_t(__builtin_ctzll(act)))
            atomicAdd(&hist[first], uint32_t(__popcll(act)));
    } else if (m) {
        atomicAdd(&hist[d], 1u);
    }
}

// Exact top-k of one row (every thread of a SEL_THREADS-thread workgroup calls it; a caller that
// selects several rows in turn puts a barrier between them).  KTH: threshold mode only (a.out_kth
// set): no winners buffer, so a cached row of up to 16K keys leaves room for two workgroups per CU.
// CACHED: the row's keys are copied to s_row (LDS) first.
template <bool CACHED, bool KTH>
__device__ void select_row(const SelectArgs& a, uint32_t row, uint32_t* s_row) {
    __shared__ uint32_t hist[256];
    __shared__ uint32_t s_digit, s_before, s_bin, s_cnt;
    __shared__ uint32_t okey[KTH ? 1 : SEL_BUF];
    __shared__ uint32_t oid[KTH ? 1 : SEL_BUF];
    __shared__ uint32_t whist[2048];     // one-pass histogram of keys below 2^11
    const int tid = threadIdx.x;
    const uint32_t orow = a.row_map ? a.row_map[row] : row;

    RowView<CACHED> rv;
    rv.keys = a.keys + int64_t(row) * a.ld;
    rv.ids = a.ids ? a.ids + int64_t(row) * a.ld : nullptr;
    rv.n = a.n;
    if (a.counts) {
        const uint32_t c = a.counts[row];
        if (c > a.n || c < a.min_count) {
            // candidate list overflowed, or too short to be the whole top-k (a threshold below
            // the k-th key): listed for the exact fallback, which writes the row
            if (tid == 0 && a.overflow_count) {
                const uint32_t p = atomicAdd(a.overflow_count, 1u);
                a.overflow_rows[p] = row;
            }
            return;
        }
        rv.n = c;
    }
    const uint32_t n = rv.n;
    if (CACHED) {
        // eight independent loads per thread per round
        for (uint32_t i0 = 0; i0 < n; i0 += 8 * SEL_THREADS) {
            uint32_t v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t i = i0 + uint32_t(j * SEL_THREADS + tid);
                v[j] = i < n ? rv.keys[i] : 0u;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t i = i0 + uint32_t(j * SEL_THREADS + tid);
                if (i < n) s_row[i] = v[j];
            }
        }
        rv.keys = s_row;
        __syncthreads();
    }
    const uint32_t K = a.k < n ? a.k : n;
    // f(key) over the row; rows read from memory load eight keys per thread before using them,
    // so a long row's pass is not one load latency per key
    auto for_keys = [&](auto&& f) {
        uint32_t i = uint32_t(tid);
        if (!CACHED)
            for (; i + 7u * SEL_THREADS < n; i += 8u * SEL_THREADS) {
                uint32_t v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = rv.key(i + uint32_t(j) * SEL_THREADS);
#pragma unroll
                for (int j = 0; j < 8; ++j) f(v[j]);
            }
        for (; i < n; i += SEL_THREADS) f(rv.key(i));
    };

    uint32_t T = 0xFFFFFFFFu, Tid = 0xFFFFFFFFu;
    bool take_all = (n <= a.k);
    if (!take_all) {
        // ---- phase 1: k-th smallest key ---------------------------------------------
        uint32_t prefix = 0, mask = 0, need = K;
        uint32_t eq = 0;
        int top = 24;  // first byte pass
        if (a.key_bits <= 11) {
            // small keys: one histogram over all key values
            const uint32_t nb = 1u << a.key_bits;
            for (uint32_t b = tid; b < nb; b += SEL_THREADS) whist[b] = 0;
            __syncthreads();
            // (a sentinel key, above every real one, lands in the top bin)
            for_keys([&](uint32_t k) { hist_add(whist, true, min(k, nb - 1u)); });
            __syncthreads();
            find_bin_wide(whist, nb, need, &s_digit, &s_before, &s_bin);
            __syncthreads();
            prefix = s_digit;
            mask = 0xFFFFFFFFu;
            need -= s_before;
            eq = s_bin;
            __syncthreads();
            top = -8;  // no byte passes left
        }
        for (int shift = top; shift >= 0; shift -= 8) {
            hist[tid] = 0;
            __syncthreads();
            for_keys([&](uint32_t k) { hist_add(hist, (k & mask) == prefix, (k >> shift) & 255u); });
            __syncthreads();
            find_digit(hist, need, &s_digit, &s_before, &s_bin);
            __syncthreads();
            prefix |= s_digit << shift;
            mask |= 255u << shift;
            need -= s_before;
            eq = s_bin;
            __syncthreads();
        }
        T = prefix;
        if (KTH || a.out_kth) {
            if (tid == 0) a.out_kth[orow] = T;
            return;
        }
        // ---- phase 2: among key == T take the `need` lowest ids ----------------------
        if (need < eq) {
            uint32_t ip = 0, im = 0, ineed = need;
            for (int shift = 24; shift >= 0; shift -= 8) {
                hist[tid] = 0;
                __syncthreads();
                for (uint32_t i = tid; i < n; i += SEL_THREADS) {
                    const bool t = rv.key(i) == T;
                    const uint32_t id = t ? rv.id(i) : 0u;
                    hist_add(hist, t && (id & im) == ip, (id >> shift) & 255u);
                }
                __syncthreads();
                find_digit(hist, ineed, &s_digit, &s_before, &s_bin);
                __syncthreads();
                ip |= s_digit << shift;
                im |= 255u << shift;
                ineed -= s_before;
                __syncthreads();
            }
            Tid = ip;
        }
    } else if (a.out_kth) {
        // fewer items than k: every key passes
        if (tid == 0) a.out_kth[orow] = 0xFFFFFFFFu;
        return;
    }

    // ---- phase 3: gather the winners and sort them by (key, id) -----------------------
    if constexpr (KTH) return;  // threshold launches always have out_kth (returned above)
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += SEL_THREADS) {
        const uint32_t k = rv.key(i);
        if (take_all || k < T || k == T) {
            const uint32_t id = rv.id(i);
            if (take_all || k < T || id <= Tid) {
                const uint32_t p = atomicAdd(&s_cnt, 1u);
                if (p < SEL_BUF) {
                    okey[p] = k;
                    oid[p] = id;
                }
            }
        }
    }
    __syncthreads();
    uint32_t cnt = s_cnt < SEL_BUF ? s_cnt : SEL_BUF;
    uint32_t P = 1;
    while (P < cnt) P <<= 1;
    for (uint32_t i = cnt + tid; i < P; i += SEL_THREADS) {
        okey[i] = 0xFFFFFFFFu;
        oid[i] = 0xFFFFFFFFu;
    }
    __syncthreads();
    for (uint32_t size = 2; size <= P; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t t = tid; t < P / 2; t += SEL_THREADS) {
                const uint32_t i = 2 * t - (t & (stride - 1));
                const uint32_t j = i + stride;
                const bool asc = (i & size) == 0;
                const uint32_t ki = okey[i], kj = okey[j], ii = oid[i], ij = oid[j];
                const bool gt = (ki > kj) || (ki == kj && ii > ij);
                if (gt == asc) {
                    okey[i] = kj;
                    okey[j] = ki;
                    oid[i] = ij;
                    oid[j] = ii;
                }
            }
            __syncthreads();
        }
    }
    // ---- write k slots -----------------------------------------------------------------
    for (uint32_t r = tid; r < a.k; r += SEL_THREADS) {
        const int64_t o = int64_t(orow) * (a.out_ld ? a.out_ld : int64_t(a.k)) + r;
        const bool have = r < cnt && r < K && okey[r] != kAbsentKey;
        const uint32_t k = have ? okey[r] : 0xFFFFFFFFu;
        if (a.out_idx) a.out_idx[o] = have ? oid[r] + a.id_offset : kSentinel;
        if (a.out_key) a.out_key[o] = k;
        if (a.out_f) {
            float v;
            if (!have) v = (a.key_kind == 1) ? -__builtin_inff() : __builtin_inff();
            else v = (a.key_kind == 1) ? float_of_key_desc(k) : float_of_key(k);
            a.out_f[o] = v;
        }
        if (a.out_i32) a.out_i32[o] = have ? (a.key_kind == 3 ? int32_t(k) : i32_of_key(k)) : INT32_MAX;
    }
}

}  // namespace va
