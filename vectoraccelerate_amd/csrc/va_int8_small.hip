// va_int8_small.hip — the int8 scan of batches of at most 128 queries (and of larger ones whose rows
// the resident-query scans do not take, 128 at a time).
//
// Streaming the codes from HBM is the cost of such a batch (10M x 512: 0.9 ms at the card's read
// rate), not the MFMA: the tiled kernel it replaces moved the rows through registers into LDS a
// stage at a time, one stage ahead.  Here the (padded) queries sit in LDS and every wave is an
// independent worker without a barrier: a tile of 16 MB rows is loaded straight into registers, all
// NCH 128-byte chunks of it, and as soon as a chunk's MFMAs are issued its registers take the same
// chunk of the wave's next tile, so NCH - 1 chunks are always in flight, across tiles.  Lane
// (r, g) = (lane % 16, lane / 16) loads 16 bytes of its row per 64-byte k-step, the four lanes of a
// row 64 contiguous bytes; v_mfma_i32_16x16x64_i8 over 16 NQB queries.  Rows need D % 4 == 0 only: the
// load that would run past the end of a row takes its last 16 bytes instead, and the query side
// holds zeros for the bytes that an earlier load already covered.
// Measured, whole searches, top-10, the tiled kernel -> here (codes at 5.66 TB/s): 10M x 512, Q = 1
// 1,402 -> 870 us, 32 1,469 -> 940, 128 1,673 -> 1,082 (905); 10M x 128, Q = 32 809 -> 281 (226);
// 4M x 200, Q = 32 2,084 -> 238 (141); 4M x 768, Q = 64 735 -> 611 (543).
#include <algorithm>

#include "va_int8.hpp"

namespace va {
namespace {

typedef int i32x4s __attribute__((ext_vector_type(4)));

constexpr uint32_t kThreads = 512, kWaves = kThreads / 64;
constexpr uint32_t kMaxD = 1024, kMaxQueries = 128;

// queries in LDS: fragment (k-step s, block n) at ((s * NQB + n) * 64 + lane) * 16
template <int NCH, int NQB>
constexpr size_t lds_bytes() {
    return size_t(2 * NCH) * NQB * 1024;
}

template <int NCH, int MB, int NQB, bool FILTER>
__global__ __launch_bounds__(kThreads, 2) void i8_small_kernel(I8Args a) {
    extern __shared__ __attribute__((aligned(16))) char qlds[];
    constexpr int KS = 2 * NCH;           // 64-byte k-steps
    constexpr uint32_t TN = 16 * MB;      // rows per wave tile
    const uint32_t tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t D = a.D, q0 = blockIdx.y * kMaxQueries;
    // ---- queries -> LDS: lane's 16 bytes of query 16n + r16 at k-step s
    for (uint32_t f = wave; f < uint32_t(KS * NQB); f += kWaves) {
        const uint32_t s = f / NQB, n = f % NQB, q = q0 + 16 * n + r16;
        const uint32_t d = 64 * s + 16 * g, d0 = min(d, D - 16);  // bytes [d0, d0 + 16), those before d zero
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t e = d0 + 4 * j;  // (4-byte groups: d, D and d0 are multiples of 4)
            w[j] = (q < a.Q && d < D && e >= d) ? *reinterpret_cast<const uint32_t*>(a.q + int64_t(q) * a.ldq + e) : 0u;
        }
        *reinterpret_cast<uint4*>(qlds + f * 1024 + lane * 16) = uint4{w[0], w[1], w[2], w[3]};
    }
    __syncthreads();
    const uint32_t ntiles = (a.N + TN - 1) / TN, step = gridDim.x * kWaves;
    // the least dot that passes: key(-dot) <= thr  <=>  -dot <= t  <=>  dot >= -t
    int32_t cut[NQB];
#pragma unroll
    for (int n = 0; n < NQB; ++n) {
        const uint32_t q = q0 + 16 * n + r16;
        cut[n] = INT32_MAX;  // (no dot of D <= 1024 codes reaches it)
        if (FILTER && q < a.Q) {
            const int64_t t = -int64_t(i32_of_key(a.thr[q]));
            cut[n] = int32_t(min(t, int64_t(INT32_MAX)));
        }
    }
    uint32_t off[KS];  // of the lane's 16 bytes in its row (rows past the tile: skipped through row_off)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const uint32_t d = 64 * s + 16 * g;
        off[s] = d < D ? min(d, D - 16) : kDmaSkip;
    }
    i32x4s rows[KS][MB];
    // chunk c of tile t into its registers (tiles past the end: nothing is read)
    auto load = [&](uint32_t t, int c) {
        const uint32_t rs = t < ntiles ? t * TN : 0u, rc = t < ntiles ? min(TN, a.N - rs) : 0u;
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<int8_t*>(a.x + int64_t(rs) * a.ldx), 0, rc ? int(uint32_t(rc - 1) * uint32_t(a.ldx) + D) : 0,
            0x00020000);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const uint32_t r = 16 * m + r16, o = off[2 * c + i];
                rows[2 * c + i][m] = __builtin_bit_cast(
                    i32x4s, __builtin_amdgcn_raw_buffer_load_b128(
                                xr, (r < rc && o != kDmaSkip) ? r * uint32_t(a.ldx) + o : kDmaSkip, 0, 0));
            }
    };
    uint32_t tile = blockIdx.x * kWaves + wave;
#pragma unroll
    for (int c = 0; c < NCH; ++c) load(tile, c);
    for (; tile < ntiles; tile += step) {
        i32x4s acc[MB][NQB];
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int n = 0; n < NQB; ++n) acc[m][n] = i32x4s{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int s = 2 * c + i;
#pragma unroll
                for (int n = 0; n < NQB; ++n) {
                    const i32x4s qf = *reinterpret_cast<const i32x4s*>(qlds + (s * NQB + n) * 1024 + lane * 16);
#pragma unroll
                    for (int m = 0; m < MB; ++m)
                        acc[m][n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(rows[s][m], qf, acc[m][n], 0, 0, 0);
                }
            }
            load(tile + step, c);
            __builtin_amdgcn_sched_barrier(0);
        }
        // lane (r16, g): query q0 + 16n + r16 against rows 16m + 4g + v in acc[m][n][v]
        const uint32_t rs = tile * TN, rc = min(TN, a.N - rs);
#pragma unroll
        for (int n = 0; n < NQB; ++n) {
            const uint32_t q = q0 + 16 * n + r16;
            if (FILTER) {
                int32_t mx = acc[0][n][0];
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int v = 0; v < 4; ++v) mx = max(mx, acc[m][n][v]);
                if (!__ballot(mx >= cut[n])) continue;
                uint32_t pass = 0;
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        pass |= uint32_t((acc[m][n][v] >= cut[n]) & (16u * m + 4u * g + v < rc)) << (4 * m + v);
                if (q >= a.Q) pass = 0;
                // one atomic for the four lanes of a query, their places in lane order (four of them: 17,557 x
                // 36, Q = 658, k = 1000 488 us a search, 155 with one)
                const uint32_t c = uint32_t(__popc(pass));
                const uint32_t c16 = uint32_t(__shfl_xor(int(c), 16)), pair = c + c16;
                const uint32_t other = uint32_t(__shfl_xor(int(pair), 32));
                uint32_t pos = 0;
                if (g == 0 && pair + other) pos = atomicAdd(a.cnt + q, pair + other);
                pos = uint32_t(__shfl(int(pos), int(r16))) + (g & 1 ? c16 : 0u) + (g & 2 ? other : 0u);
                if (!pass) continue;
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        if (!((pass >> (4 * m + v)) & 1u)) continue;
                        if (pos < a.cap) {
                            const int64_t o = int64_t(q) * a.cap + pos;
                            a.cand_key[o] = key_of_i32(-acc[m][n][v]);
                            a.cand_id[o] = rs + 16 * m + 4 * g + v;
                        }
                        ++pos;
                    }
            } else if (q < a.Q) {
                uint32_t* o = a.out_k + int64_t(q) * a.ldo + rs;
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const uint32_t r = 16 * m + 4 * g + v;
                        if (r < rc) o[r] = key_of_i32(-acc[m][n][v]);
                    }
            }
        }
    }
}

template <int NCH, int MB, int NQB>
va_status go(va_context* ctx, const I8Args& a, bool filter) {
    const uint32_t tiles = (a.N + 16 * MB - 1) / (16 * MB);
    constexpr size_t lds = lds_bytes<NCH, NQB>();
    const uint32_t grid = std::max<uint32_t>(1, std::min((tiles + kWaves - 1) / kWaves, uint32_t(ctx->num_cus)));
    auto kern = filter ? &i8_small_kernel<NCH, MB, NQB, true> : &i8_small_kernel<NCH, MB, NQB, false>;
    if (lds > 48 * 1024)
        VA_CHECK_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    kern<<<dim3(grid, (a.Q + kMaxQueries - 1) / kMaxQueries), dim3(kThreads), lds, ctx->stream>>>(a);
    VA_CHECK_LAUNCH(ctx);
    return VA_OK;
}

// 16, 32, 64 or 128 queries; fewer row blocks where the accumulators and the tile's registers would
// not leave two waves per SIMD.
template <int NCH, int MB>
va_status go_q(va_context* ctx, const I8Args& a, bool filter) {
    if (a.Q <= 16) return go<NCH, MB, 1>(ctx, a, filter);
    if (a.Q <= 32) return go<NCH, MB, 2>(ctx, a, filter);
    if (a.Q <= 64) return go<NCH, MB, 4>(ctx, a, filter);
    return go<NCH, (NCH <= 4 ? (MB > 2 ? 2 : MB) : 1), 8>(ctx, a, filter);
}

}  // namespace

bool i8_small_ok(const I8Args& a) {
    return !a.qrow && a.Q <= kMaxQueries * 65535u && a.D >= 16 && a.D <= kMaxD && a.D % 4 == 0 && a.ldq % 4 == 0 && a.ldx % 4 == 0 &&
           ((reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.x)) & 3) == 0 &&
           uint64_t(63) * uint64_t(a.ldx) + a.D <= kDmaMaxBytes && a.N <= 0xFFFF0000u;
}

va_status launch_i8_small(va_context* ctx, const I8Args& a, bool filter) {
    if (a.D <= 128) return go_q<1, 4>(ctx, a, filter);
    if (a.D <= 256) return go_q<2, 4>(ctx, a, filter);
    if (a.D <= 512) return go_q<4, 2>(ctx, a, filter);
    if (a.D <= 768) return go_q<6, 2>(ctx, a, filter);
    return go_q<8, 1>(ctx, a, filter);
}

}  // namespace va
