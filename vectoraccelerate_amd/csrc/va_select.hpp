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
constexpr uint32_t SEL_FEW = 128;   // items ranked by comparing all pairs
constexpr uint32_t SEL_BITS = 11, SEL_BINS = 1u << SEL_BITS;  // bits and bins of one histogram pass

template <bool CACHED>
struct RowView {
    const uint32_t* keys;  // the row in memory, or its copy in LDS
    const uint32_t* ids;
    uint32_t n;
    __device__ uint32_t key(uint32_t i) const { return keys[i]; }
    __device__ uint32_t id(uint32_t i) const { return ids ? ids[i] : i; }
};

// The LDS of a search for the k-th smallest value.
struct RadixLds {
    uint32_t digit, before, bin, cnt, lo, hi;
    uint32_t wsum[16];
    uint32_t whist[SEL_BINS];
};
// ... and of a row's selection (KTH: threshold mode, without the winners).
template <bool KTH>
struct SelectLds : RadixLds {
    uint32_t okey[KTH ? 1 : SEL_BUF];
    uint32_t oid[KTH ? 1 : SEL_BUF];
};

// The bin of a histogram of nb <= 2048 bins holding the need-th item: each thread sums a
// few bins, a block-wide scan of the sums, then the thread whose range holds the item finds it.
template <int NT>
__device__ inline void find_bin_wide(const uint32_t* hist, uint32_t nb, uint32_t need, uint32_t* wsum,
                                     uint32_t* s_digit, uint32_t* s_before, uint32_t* s_bin) {
    constexpr int PER = int(SEL_BINS) / NT;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const uint32_t b = uint32_t(tid) * PER + i;
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
        for (int i = 0; i < PER; ++i) {
            if (run < need && need <= run + c[i]) {
                *s_digit = uint32_t(tid) * PER + i;
                *s_before = run;
                *s_bin = c[i];
            }
            run += c[i];
        }
    }
}

// Adds this lane's item to bin d of the histogram when m.  Keys of one search crowd into few bins
// (ties, excluded rows, Hamming distances), and 64 lanes incrementing one LDS word serialise: the
// bin of the first lane, and where eight lanes or more share it that of the first one left, are each
// added once for all lanes that share them, the rest one by one.
__device__ __forceinline__ void hist_add(uint32_t* hist, bool m, uint32_t d) {
    uint64_t rest = __ballot(m);
    const uint32_t lane = threadIdx.x & 63;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        if (!rest) return;
        const int l = __builtin_ctzll(rest);
        const uint32_t f = uint32_t(__builtin_amdgcn_readlane(int(d), l));
        const uint64_t same = __ballot(m && d == f) & rest;
        if (lane == uint32_t(l)) atomicAdd(&hist[f], uint32_t(__popcll(same)));
        rest &= ~same;
        if (__popcll(same) < 8) break;
    }
    if ((rest >> lane) & 1ull) atomicAdd(&hist[d], 1u);
}

// The need-th smallest of the few <= SEL_FEW values in lds.whist; need and eq as radix_kth's.  (The
// loop's reads are independent: unrolled, they are not one LDS latency each.)
__device__ inline uint32_t kth_of_few(RadixLds& lds, uint32_t few, uint32_t& need, uint32_t& eq) {
    const uint32_t tid = threadIdx.x, want = need;
    if (tid < few) {
        const uint32_t v = lds.whist[tid];
        uint32_t below = 0, same = 0;
#pragma unroll 8
        for (uint32_t j = 0; j < few; ++j) {
            const uint32_t o = lds.whist[j];
            below += o < v;
            same += o == v;
        }
        if (below < want && want <= below + same) {  // (every item equal to the answer writes the same)
            lds.lo = v;
            lds.before = below;
            lds.bin = same;
        }
    }
    __syncthreads();
    const uint32_t t = lds.lo;
    need = want - lds.before;
    eq = lds.bin;
    __syncthreads();
    return t;
}

// The need-th smallest value of the items for_vals(f) runs f(value, taken) over, all within
// [base, base + 2^bits): histograms of up to 11 bits at a time, from the top, until the bin that
// holds it has at most SEL_FEW items (the tail of a spread of distances: usually after the
// first), which are ranked directly; eq, the number of items taken, at once where that few.  need
// becomes its rank among the items equal to it, eq their number.  Every thread of an NT-thread
// workgroup calls it.
template <int NT, class ForVals>
__device__ inline uint32_t radix_kth(RadixLds& lds, ForVals&& for_vals, uint32_t base, uint32_t bits, uint32_t& need,
                                     uint32_t& eq) {
    const int tid = threadIdx.x;
    uint32_t prefix = 0;
    uint32_t left = bits;
    // (1,024 threads are for long rows: there the path would only cost registers, and past 80 SGPRs a CU
    // holds one such workgroup instead of two)
    if (NT <= 256 && left && eq <= SEL_FEW) {
        if (tid == 0) lds.cnt = 0;
        __syncthreads();
        for_vals([&](uint32_t v, bool taken) {
            if (taken) lds.whist[atomicAdd(&lds.cnt, 1u)] = v;
        });
        __syncthreads();
        return kth_of_few(lds, eq, need, eq);
    }
    while (left) {
        const uint32_t w = left < SEL_BITS ? left : SEL_BITS, sh = left - w, nb = 1u << w;
        for (uint32_t b = tid; b < nb; b += NT) lds.whist[b] = 0;
        __syncthreads();
        for_vals([&](uint32_t v, bool taken) {
            const uint32_t d = v - base;
            const bool m = taken && (left == bits || (d >> left) == prefix);
            // (a value past the range, a sentinel above every real one, lands in the top bin)
            const uint32_t bin = d >> sh;
            hist_add(lds.whist, m, left == bits ? min(bin, nb - 1u) : (bin & (nb - 1u)));
        });
        __syncthreads();
        find_bin_wide<NT>(lds.whist, nb, need, lds.wsum, &lds.digit, &lds.before, &lds.bin);
        __syncthreads();
        prefix = (prefix << w) | lds.digit;
        need -= lds.before;
        eq = lds.bin;
        left = sh;
        __syncthreads();
        if (left && eq <= SEL_FEW) {
            if (tid == 0) lds.cnt = 0;
            __syncthreads();
            for_vals([&](uint32_t v, bool taken) {
                if (taken && ((v - base) >> left) == prefix) lds.whist[atomicAdd(&lds.cnt, 1u)] = v;
            });
            __syncthreads();
            return kth_of_few(lds, eq, need, eq);
        }
    }
    return base + prefix;
}

// The need-th smallest key of for_keys(f): mn and mx are the smallest and largest of this thread's
// keys.  The histograms start below the leading bits that all keys share: nearby distances have
// equal top bits, and bins of those bits alone would count everything in one bin.  The smallest key
// needs none (eq is then left at "more than one": its ties were not counted).
template <int NT, class ForKeys>
__device__ inline uint32_t kth_key(RadixLds& lds, ForKeys&& for_keys, uint32_t mn, uint32_t mx, uint32_t& need,
                                   uint32_t& eq) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mn = min(mn, uint32_t(__shfl_xor(int(mn), off)));
        mx = max(mx, uint32_t(__shfl_xor(int(mx), off)));
    }
    if (threadIdx.x == 0) {
        lds.lo = 0xFFFFFFFFu;
        lds.hi = 0;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&lds.lo, mn);
        atomicMax(&lds.hi, mx);
    }
    __syncthreads();
    const uint32_t lo = lds.lo, hi = lds.hi;
    if (need == 1) {
        eq = 2;
        return lo;
    }
    return radix_kth<NT>(lds, [&](auto&& f) { for_keys([&](uint32_t k) { f(k, true); }); }, lo,
                         hi == lo ? 0u : 32u - uint32_t(__builtin_clz(hi - lo)), need, eq);
}

// Exact top-k of one row (every thread of an NT-thread workgroup calls it; a caller that selects
// several rows in turn puts a barrier between them).  KTH: threshold mode only (a.out_kth
// set): no winners buffer, so a cached row of up to 16K keys leaves room for two workgroups per CU.
// CACHED: the row's keys are copied to s_row (LDS) first.  Inlined by force: a call copies a (232
// bytes) to each lane's private memory, also in a fallback that finds nothing to do.
template <int NT, bool CACHED, bool KTH>
__device__ __forceinline__ void select_row(const SelectArgs& a, uint32_t row, SelectLds<KTH>& lds, uint32_t* s_row) {
    uint32_t& s_cnt = lds.cnt;
    uint32_t *const okey = lds.okey, *const oid = lds.oid;
    const int tid = threadIdx.x;
    const uint32_t orow = a.row_map ? a.row_map[row] : row;

    RowView<CACHED> rv;
    uint32_t id_offset = a.id_offset;
    if (a.nseg) {
        // segment row % nseg of dense row row / nseg
        const uint32_t s0 = (row % a.nseg) * a.seg;
        rv.keys = a.keys + int64_t(row / a.nseg) * a.ld + s0;
        rv.ids = nullptr;
        rv.n = min(a.seg, a.n - s0);
        id_offset += s0;
    } else {
        rv.keys = a.keys + int64_t(row) * a.ld;
        rv.ids = a.ids ? a.ids + int64_t(row) * a.ld : nullptr;
        rv.n = a.n;
    }
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
    uint32_t mn = 0xFFFFFFFFu, mx = 0;  // of this thread's keys
    if (CACHED) {
        // eight independent loads per thread per round
        for (uint32_t i0 = 0; i0 < n; i0 += 8 * NT) {
            uint32_t v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t i = i0 + uint32_t(j * NT + tid);
                v[j] = i < n ? rv.keys[i] : 0u;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t i = i0 + uint32_t(j * NT + tid);
                if (i < n) {
                    s_row[i] = v[j];
                    mn = min(mn, v[j]);
                    mx = max(mx, v[j]);
                }
            }
        }
        rv.keys = s_row;
        __syncthreads();
    }
    const uint32_t K = a.k < n ? a.k : n;
    // f(key, i) over the row; rows read from memory load eight keys per thread before using them,
    // so a long row's pass is not one load latency per key
    auto for_keys = [&](auto&& f) {
        uint32_t i = uint32_t(tid);
        if (!CACHED)
            for (; i + 7u * NT < n; i += 8u * NT) {
                uint32_t v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = rv.key(i + uint32_t(j) * NT);
#pragma unroll
                for (int j = 0; j < 8; ++j) f(v[j], i + uint32_t(j) * NT);
            }
        for (; i < n; i += NT) f(rv.key(i), i);
    };

    uint32_t T = 0xFFFFFFFFu, Tid = 0xFFFFFFFFu;
    bool take_all = (n <= a.k);
    if (!take_all) {
        // ---- phase 1: k-th smallest key ---------------------------------------------
        uint32_t need = K, eq = n;
        if (a.key_bits <= SEL_BITS) {
            T = radix_kth<NT>(lds, [&](auto&& f) { for_keys([&](uint32_t k, uint32_t) { f(k, true); }); }, 0u, a.key_bits,
                              need, eq);
        } else {
            // A row read from memory: a pass for its keys' range pays where they lie close together, as
            // distances and the winners of segments do (a sample of 20,000 L2^2 distances, 200 queries:
            // 14 us, 19 without).  A caller's values may lie anywhere and start from the top bits (3,000
            // rows of 30,000 N(0, 1) values, k = 600: 589 us, 648 with it).
            if (!CACHED && a.spread && K > 1) {
                mn = 0u;
                mx = 0xFFFFFFFFu;
            } else if (!CACHED) {
                for_keys([&](uint32_t k, uint32_t) {
                    mn = min(mn, k);
                    mx = max(mx, k);
                });
            }
            T = kth_key<NT>(lds, [&](auto&& f) { for_keys([&](uint32_t k, uint32_t) { f(k); }); }, mn, mx, need, eq);
        }
        if (KTH || a.out_kth) {
            if (tid == 0) a.out_kth[orow] = T;
            return;
        }
        // ---- phase 2: among key == T take the `need` lowest ids ----------------------
        if (need < eq && need == 1) {  // the lowest id
            for_keys([&](uint32_t k, uint32_t i) {
                if (k == T) Tid = min(Tid, rv.id(i));
            });
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) Tid = min(Tid, uint32_t(__shfl_xor(int(Tid), off)));
            __syncthreads();  // (lds.lo may still be read)
            if (tid == 0) lds.lo = 0xFFFFFFFFu;
            __syncthreads();
            if ((tid & 63) == 0) atomicMin(&lds.lo, Tid);
            __syncthreads();
            Tid = lds.lo;
        } else if (need < eq)
            Tid = radix_kth<NT>(
                lds,
                [&](auto&& f) {
                    for_keys([&](uint32_t k, uint32_t i) {
                        const bool t = k == T;
                        f(t ? rv.id(i) : 0u, t);
                    });
                },
                0u, rv.ids ? 32u : 32u - uint32_t(__builtin_clz(n - 1)), need, eq);  // (columns: below n)
    } else if (a.out_kth) {
        // fewer items than k: every key passes
        if (tid == 0) a.out_kth[orow] = 0xFFFFFFFFu;
        return;
    }

    // ---- phase 3: gather the winners and sort them by (key, id) -----------------------
    if constexpr (KTH) return;  // threshold launches always have out_kth (returned above)
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    for_keys([&](uint32_t k, uint32_t i) {
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
    });
    __syncthreads();
    const uint32_t cnt = s_cnt < SEL_BUF ? s_cnt : SEL_BUF;
    // slot r of the output: winner (wk, wid), or missing
    auto put = [&](uint32_t r, bool have, uint32_t wk, uint32_t wid) {
        const int64_t o = int64_t(orow) * (a.out_ld ? a.out_ld : int64_t(a.k)) + r;
        have = have && wk != kAbsentKey;
        const uint32_t k = have ? wk : 0xFFFFFFFFu;
        if (a.out_idx) a.out_idx[o] = !have ? kSentinel : a.out_map ? a.out_map[wid + id_offset] : wid + id_offset;
        if (a.out_key) a.out_key[o] = k;
        if (a.out_f) {
            float v;
            if (!have) v = (a.key_kind == 1) ? -__builtin_inff() : __builtin_inff();
            else v = (a.key_kind == 1) ? float_of_key_desc(k) : float_of_key(k);
            a.out_f[o] = v;
        }
        if (a.out_i32) a.out_i32[o] = have ? (a.key_kind == 3 ? int32_t(k) : i32_of_key(k)) : INT32_MAX;
    };
    if (cnt <= SEL_FEW) {
        // few winners: each finds its slot by comparing itself with all of them
        if (uint32_t(tid) < cnt) {
            // (no branches in the loop: its reads then go out together, not one LDS latency each)
            const uint32_t wk = okey[tid], wid = oid[tid];
            const uint64_t w = uint64_t(wk) << 32 | wid;
            uint32_t r = 0;
#pragma unroll 8
            for (uint32_t j = 0; j < cnt; ++j) {
                const uint64_t o = uint64_t(okey[j]) << 32 | oid[j];
                r += uint32_t(o < w) + (uint32_t(o == w) & uint32_t(j < uint32_t(tid)));
            }
            if (r < K) put(r, true, wk, wid);
        }
        for (uint32_t r = min(cnt, K) + tid; r < a.k; r += NT) put(r, false, 0, 0);
        return;
    }
    uint32_t P = 1;
    while (P < cnt) P <<= 1;
    for (uint32_t i = cnt + tid; i < P; i += NT) {
        okey[i] = 0xFFFFFFFFu;
        oid[i] = 0xFFFFFFFFu;
    }
    __syncthreads();
    for (uint32_t size = 2; size <= P; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t t = tid; t < P / 2; t += NT) {
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
    for (uint32_t r = tid; r < a.k; r += NT) put(r, r < cnt && r < K, okey[r < cnt ? r : 0], oid[r < cnt ? r : 0]);
}

}  // namespace va
