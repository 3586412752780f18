// va_dist.hip — fp32 distance GEMM on CDNA4 MFMA (v_mfma_f32_32x32x2_f32).
//
// One kernel computes every Q x N distance family of the search path:
//   dist(q, x) from the contraction q.x and the squared norms |q|^2, |x|^2, where the
//   norms are accumulated on the VALU from the same LDS fragments that feed the MFMA
//   (no separate norm pass over the database).
// Replaces the reference's per-pair scalar loops: l2_distance_kernel
// (Metal/Shaders/L2Distance.metal:34-91), dot_product_kernel (DotProduct.metal:29-96) and the
// distance loop of fused_l2_topk (AdvancedTopK.metal:238-242).
//
// Tile geometry (256 threads = 4 wave64):
//   wave tile      = 32 queries x 128 database rows = 4 MFMA blocks of 32x32, 64 acc/lane
//   workgroup tile = (32*WQ) queries x (128*WN) rows, WQ*WN = 4
//   K loop         = LDS stages of KC=16 d-values, double buffered, one barrier per stage
// MFMA operand map: A = database rows (M), B = queries (N).  The contraction index is
// permuted so one ds_read_b128 per lane feeds four MFMA steps: at step s of an 8-wide
// d-group, lane half h supplies d = d0 + 4h + s for both A and B.
// Output map of a 32x32 block (lane l, acc v): row m = 8*(v/4) + 4*(l/32) + v%4,
// column n = l%32 — so each lane owns ONE query and 64 database rows.
#include <cfloat>

#include <algorithm>

#include "va_distop.hpp"
#include "va_internal.hpp"

namespace va {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int KC = 16;               // d-values per LDS stage
#ifndef VA_DIST_SWZ
#define VA_DIST_SWZ 1
#endif
#ifndef VA_DIST_WPE
#define VA_DIST_WPE 2      // waves per SIMD the register-staged kernel is compiled for
#endif
#ifndef VA_DIST_DMA_WPE
#define VA_DIST_DMA_WPE 4  // ... and the direct-load kernel
#endif
#ifndef VA_DIST_DMA
#define VA_DIST_DMA 1
#endif
#ifndef VA_DIST_DMA_SLOTS
#define VA_DIST_DMA_SLOTS 2  // LDS ring slots of the direct-load kernel (stages in flight + 1)
#endif
#if VA_DIST_SWZ
// 64-byte rows, unpadded: 16-byte chunk c of row r sits at chunk c ^ ((r >> 2) & 3).
// ds_read_b128 / ds_write_b128 serve 16 lanes per clock across 64 banks; the 16 rows of a
// fragment read (and the 4 x 4 chunks of a 16-lane write) land in 16 distinct bank groups.
constexpr int LDS_STRIDE = KC;
__device__ __forceinline__ int lds_chunk(int row, int c) { return c ^ ((row >> 2) & 3); }
#else
constexpr int LDS_STRIDE = KC + 4;   // 80-byte rows: conflict-free ds_read_b128 / ds_write_b128
__device__ __forceinline__ int lds_chunk(int row, int c) { return c; }
#endif

// WQ x WN waves of 64 lanes; each wave owns 32 queries x 128 rows (4 MFMA blocks).
template <int WQ, int WN>
struct Tile {
    static constexpr int NW = WQ * WN;
    static constexpr int NT = 64 * NW;
    static constexpr int TQ = 32 * WQ;
    static constexpr int TN = 128 * WN;
    static constexpr int ROWS = TQ + TN;
    static constexpr int CHUNKS = ROWS * (KC / 4);
    static constexpr int CPT = (CHUNKS + NT - 1) / NT;
    static constexpr int STAGE = ROWS * LDS_STRIDE;
    // register-staged loads: a one-wave tile keeps one LDS stage (the next stage waits in
    // registers), 44 KB instead of 87 KB, so three workgroups share a CU instead of one
    static constexpr int NSTAGE = NW == 1 ? 1 : 2;
    static constexpr size_t LDS_BYTES = size_t(NSTAGE * STAGE + NW * 128) * sizeof(float);
    // direct-to-LDS loads: 16-row groups of 1 KiB (one wave-wide load each), the same number
    // per wave (the last few may be padding), two ring slots
    static constexpr int GROUPS = ROWS / 16;
    static constexpr int GPW = (GROUPS + NW - 1) / NW;
    static constexpr int DSTAGE = GPW * NW * 256;  // floats per slot
    static constexpr size_t DMA_LDS_BYTES = size_t(VA_DIST_DMA_SLOTS * DSTAGE + NW * 128) * sizeof(float);
};

// DMA = true: the stages move global -> LDS by direct buffer loads (no register staging, so
// fewer VGPRs and more waves per SIMD); needs 16-byte rows (VEC) and the swizzled 64-byte LDS
// rows.  DMA = false: register-staged loads, any row alignment.
// One tile: queries qs + i (i < qc; through qrow when given) x database rows at positions
// rs + j (j < rc).  Every wave of the workgroup calls it with the same tile.
// LOOP: called once per iteration of the planned launch's tile loop.  The thread index then goes
// through an opaque move, so that nothing derived from it is hoisted out of the loop and held
// across the whole tile (the main loop has no register to spare).
// (the planned launches are the IVF list scans: L2^2, the distance fixed at compile time)
template <int WQ, int WN, bool VEC, int OUT, bool DMA, bool LOOP = false>
__device__ __forceinline__ void dist_tile(const DistArgs& a, uint32_t qs, uint32_t qc, uint32_t rs, uint32_t rc) {
    const int op = LOOP ? int(OP_L2SQ) : int(a.op);
    using T = Tile<WQ, WN>;
    extern __shared__ float lds[];
    float* nrm = lds + (DMA ? VA_DIST_DMA_SLOTS * T::DSTAGE : T::NSTAGE * T::STAGE);  // [waves][128] squared norms of the wave's rows

    int tid = int(threadIdx.x);
    if constexpr (LOOP) asm volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wave % WQ;
    const int wn = wave / WQ;
    const int l32 = lane & 31;
    const int hh = lane >> 5;

    f32x16 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;
    float qss = 0.0f;
    float xss[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // fragment rows start at multiples of 32, so every fragment row shares l32's chunk swizzle
    const int boff = (wq * 32 + l32) * LDS_STRIDE;
    const int aoff = (T::TQ + wn * 128 + l32) * LDS_STRIDE;
    int koff[KC / 8];
#pragma unroll
    for (int g = 0; g < KC / 8; ++g) koff[g] = 4 * lds_chunk(l32, 2 * g + hh);
    // one 16-value stage of MFMAs from an LDS slot; norms accumulate from the same fragments
    auto compute = [&](const float* st) {
#pragma unroll
        for (int g = 0; g < KC / 8; ++g) {
            const f32x4v bv = *reinterpret_cast<const f32x4v*>(st + boff + koff[g]);
            qss = fmaf(bv[0], bv[0], qss);
            qss = fmaf(bv[1], bv[1], qss);
            qss = fmaf(bv[2], bv[2], qss);
            qss = fmaf(bv[3], bv[3], qss);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const f32x4v av = *reinterpret_cast<const f32x4v*>(st + aoff + b * 32 * LDS_STRIDE + koff[g]);
                xss[b] = fmaf(av[0], av[0], xss[b]);
                xss[b] = fmaf(av[1], av[1], xss[b]);
                xss[b] = fmaf(av[2], av[2], xss[b]);
                xss[b] = fmaf(av[3], av[3], xss[b]);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[0], bv[0], acc[b], 0, 0, 0);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[1], bv[1], acc[b], 0, 0, 0);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[2], bv[2], acc[b], 0, 0, 0);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[3], bv[3], acc[b], 0, 0, 0);
            }
        }
    };
    const int nstages = int((a.D + KC - 1) / KC);
    if constexpr (DMA) {
        // 16-row group gi of a slot is rows 16*gi .. 16*gi+15 (queries first, then database
        // rows); lane L loads row 16*gi + L/4, physical chunk L%4 = logical chunk
        // (L%4) ^ swizzle(row).  Rows outside the tile and columns past D load from an offset
        // past the descriptor and land as zeros.
        // every offset below addresses a real row (checked by the launcher to stay under
        // kDmaMaxBytes), so the descriptors only need to bound kDmaSkip
        const dma_rsrc qres = make_dma_rsrc(a.q, kDmaMaxBytes);
        const dma_rsrc xres = make_dma_rsrc(a.x + int64_t(rs) * a.ldx, kDmaMaxBytes);
        uint32_t base[T::GPW], colb[T::GPW];
#pragma unroll
        for (int i = 0; i < T::GPW; ++i) {
            const int row = 16 * (wave + T::NW * i) + (lane >> 2);
            const int c = lds_chunk(row, lane & 3);
            colb[i] = uint32_t(4 * c);
            base[i] = kDmaSkip;
            if (row < T::TQ) {
                if (uint32_t(row) < qc) {
                    const uint32_t r = a.qrow ? a.qrow[qs + row] : qs + row;
                    base[i] = uint32_t(int64_t(r) * a.ldq * 4) + 16u * uint32_t(c);
                }
            } else if (row < T::ROWS) {
                const uint32_t jr = uint32_t(row - T::TQ);
                if (jr < rc) base[i] = uint32_t(int64_t(jr) * a.ldx * 4) + 16u * uint32_t(c);
            }
        }
        const uint32_t lds0 = lds_addr_of(lds);
        auto issue = [&](uint32_t d0, int slot) {
#pragma unroll
            for (int i = 0; i < T::GPW; ++i) {
                const uint32_t voff = (base[i] != kDmaSkip && d0 + colb[i] < a.D) ? base[i] + d0 * 4u : kDmaSkip;
                const int grp = wave + T::NW * i;
                lds_dma16(16 * grp < T::TQ ? qres : xres, voff,
                          lds0 + uint32_t(slot * T::DSTAGE + grp * 256) * 4u);
            }
        };
        if constexpr (VA_DIST_DMA_SLOTS == 2) {
            issue(0, 0);
            wait_vmcnt<0>();
            __syncthreads();
            for (int s = 0; s < nstages; ++s) {
                const bool more = (s + 1) < nstages;
                if (more) issue(uint32_t(s + 1) * KC, (s + 1) & 1);  // slot last read before the previous barrier
                compute(lds + (s & 1) * T::DSTAGE);
                if (more) wait_vmcnt<0>();
                __syncthreads();
            }
        } else {
            // three slots: stage s+2 loads while stage s computes
            issue(0, 0);
            if (nstages > 1) issue(KC, 1);
            int slot = 0;
            for (int s = 0; s < nstages; ++s) {
                if (s + 1 < nstages) wait_vmcnt<T::GPW>();
                else wait_vmcnt<0>();
                __syncthreads();  // stage s visible; every wave is past the reads of slot (s + 2) % 3
                if (s + 2 < nstages) issue(uint32_t(s + 2) * KC, slot == 0 ? 2 : slot - 1);
                compute(lds + slot * T::DSTAGE);
                slot = slot == 2 ? 0 : slot + 1;
            }
            __syncthreads();  // the epilogue reuses LDS only after every wave's last reads
        }
    } else {
        // source row pointers of this thread's load chunks (fixed across stages)
        const float* src[T::CPT];
        int ldsoff[T::CPT];
        uint32_t colv[T::CPT];
#pragma unroll
        for (int j = 0; j < T::CPT; ++j) {
            const int c = tid + T::NT * j;
            src[j] = nullptr;
            ldsoff[j] = -1;
            colv[j] = 0;
            if (c < T::CHUNKS) {
                const int row = c >> 2;
                const int col = (c & 3) * 4;
                ldsoff[j] = row * LDS_STRIDE + 4 * lds_chunk(row, col / 4);
                colv[j] = uint32_t(col);
                if (row < T::TQ) {
                    if (uint32_t(row) < qc) {
                        const uint32_t r = a.qrow ? a.qrow[qs + row] : qs + row;
                        src[j] = a.q + int64_t(r) * a.ldq + col;
                    }
                } else {
                    const uint32_t jr = uint32_t(row - T::TQ);
                    if (jr < rc) {
                        const int64_t xr = a.gather ? int64_t(a.gather[int64_t(qs) * a.gcap + rs + jr])
                                                    : int64_t(rs + jr);
                        src[j] = a.x + xr * a.ldx + col;
                    }
                }
            }
        }

        f32x4v pre[T::CPT];
        auto load = [&](uint32_t d0) {
#pragma unroll
            for (int j = 0; j < T::CPT; ++j) {
                f32x4v v = {0.0f, 0.0f, 0.0f, 0.0f};
                const uint32_t d = d0 + colv[j];
                if (src[j]) {
                    if (VEC) {
                        if (d < a.D) v = *reinterpret_cast<const f32x4v*>(src[j] + d0);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (d + e < a.D) v[e] = src[j][d0 + e];
                    }
                }
                pre[j] = v;
            }
        };
        auto store = [&](float* stage) {
#pragma unroll
            for (int j = 0; j < T::CPT; ++j)
                if (ldsoff[j] >= 0) *reinterpret_cast<f32x4v*>(stage + ldsoff[j]) = pre[j];
        };

        load(0);
        store(lds);
        __syncthreads();
        for (int s = 0; s < nstages; ++s) {
            const bool more = (s + 1) < nstages;
            if (more) load(uint32_t(s + 1) * KC);
            if constexpr (T::NSTAGE == 1) {
                compute(lds);
                __syncthreads();  // every read of the stage is done before it is overwritten
                if (more) store(lds);
            } else {
                compute(lds + (s & 1) * T::STAGE);
                if (more) store(lds + ((s + 1) & 1) * T::STAGE);
            }
            __syncthreads();
        }
    }

    // combine the two lane halves of every partial sum of squares
    const float qq = qss + __shfl_xor(qss, 32);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const float t = xss[b] + __shfl_xor(xss[b], 32);
        if (hh == 0) nrm[wave * 128 + b * 32 + l32] = t;
    }
    __syncthreads();

    const uint32_t li = uint32_t(wq * 32 + l32);  // query slot of this lane in the tile
    if (li >= qc) return;
    const uint32_t orow = qs + li;                                   // dense output row
    if (OUT == OUT_ARGMIN) {
        // the lane's 64 rows in increasing id order, strict < : ties keep the lower row id; the two
        // lane halves hold the same query and the other rows of each 8-row group
        uint32_t bk = 0xFFFFFFFFu, bi = 0xFFFFFFFFu;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int mloc = b * 32 + 8 * j + 4 * hh;
                const f32x4v xx = *reinterpret_cast<const f32x4v*>(nrm + wave * 128 + mloc);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t r = uint32_t(wn * 128 + mloc + e);
                    const uint32_t key = key_of_float(apply_op(op, acc[b][4 * j + e], qq, xx[e]));
                    if (r < rc && key < bk && key < 0xFFFFFFFEu) {  // NaN distances never win
                        bk = key;
                        bi = rs + r;
                    }
                }
            }
        unsigned long long best = (static_cast<unsigned long long>(bk) << 32) | bi;
        const unsigned long long other =
            (static_cast<unsigned long long>(uint32_t(__shfl_xor(int(bk), 32))) << 32) | uint32_t(__shfl_xor(int(bi), 32));
        best = other < best ? other : best;
        if (hh == 0 && best != ~0ull) atomicMin(a.best + orow, best);
        return;
    }
    const uint32_t qi = (OUT == OUT_FILTER && a.qrow) ? a.qrow[orow] : orow;  // query id (filter)
    if (OUT == OUT_FILTER) {
        const uint32_t thr = a.thr[qi];
        // Keys of passing values are reserved with one atomic and written; the direct-load
        // kernel does this for half of the lane's 64 values at a time, which keeps its
        // epilogue within the main loop's 128-VGPR budget (4 waves per SIMD).
        constexpr int HALVES = DMA ? 2 : 1;
        constexpr int NB = 4 / HALVES;  // MFMA blocks per half
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
            uint64_t pass = 0;  // bit 16(b - NB h) + 4j + e
            uint32_t keys[16 * NB];
#pragma unroll
            for (int bb = 0; bb < NB; ++bb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int b = NB * h + bb;
                    const int mloc = b * 32 + 8 * j + 4 * hh;
                    const f32x4v xx = *reinterpret_cast<const f32x4v*>(nrm + wave * 128 + mloc);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t key = key_of_float(apply_op(op, acc[b][4 * j + e], qq, xx[e]));
                        keys[16 * bb + 4 * j + e] = key;
                        const bool p = (uint32_t(wn * 128 + mloc + e) < rc) & (key <= thr);
                        pass |= uint64_t(p) << (16 * bb + 4 * j + e);
                    }
                }
            if (!pass) continue;
            uint32_t pos = atomicAdd(a.cnt + qi, uint32_t(__popcll(pass)));
#pragma unroll
            for (int t = 0; t < 16 * NB; ++t) {
                if (!((pass >> t) & 1)) continue;
                if (pos < a.cap) {
                    const int b = NB * h + (t >> 4), j = (t >> 2) & 3, e = t & 3;
                    const uint32_t p = rs + uint32_t(wn * 128 + b * 32 + 8 * j + 4 * hh + e);
                    const int64_t o = int64_t(qi) * a.cap + pos;
                    a.cand_key[o] = keys[t];
                    a.cand_id[o] = a.ids ? a.ids[p] : a.id_base + p;
                }
                ++pos;
            }
        }
        return;
    }

#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int mloc = b * 32 + 8 * j + 4 * hh;
            const f32x4v xx = *reinterpret_cast<const f32x4v*>(nrm + wave * 128 + mloc);
            float val[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) val[e] = apply_op(op, acc[b][4 * j + e], qq, xx[e]);
            const uint32_t jr = uint32_t(wn * 128 + mloc);  // row slot of acc element e = 0
            if (OUT == OUT_KEYS) {
                uint32_t* o = a.out_k + int64_t(orow) * a.ldo + rs + jr;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (jr + e < rc) o[e] = key_of_float(val[e]);
            } else {
                float* o = a.out_f + int64_t(orow) * a.ldo + rs + jr;
                if (jr + 3 < rc && ((a.ldo & 3) == 0) && ((reinterpret_cast<uintptr_t>(o) & 15) == 0)) {
                    f32x4v w = {val[0], val[1], val[2], val[3]};
                    *reinterpret_cast<f32x4v*>(o) = w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (jr + e < rc) o[e] = val[e];
                }
            }
        }
    }
}

// PLAN: a device-planned list-major launch (a.plan): a fixed grid loops over the tiles of the
// plan, each decoded from the plan's per-list tile counts.
template <int WQ, int WN, bool VEC, int OUT, bool DMA, bool PLAN>
__global__ __launch_bounds__(64 * WQ * WN, DMA ? VA_DIST_DMA_WPE : VA_DIST_WPE) void dist_gemm_kernel(DistArgs a) {
    using T = Tile<WQ, WN>;
    static_assert(!DMA || (VEC && LDS_STRIDE == KC), "direct loads need 16-byte rows and unpadded LDS rows");
    if constexpr (PLAN) {
        const uint32_t total = a.plan.pre[a.plan.C];
        for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
            uint32_t qs, qc, rs, rc;
            plan_tile(a.plan, t, uint32_t(T::TQ), uint32_t(T::TN), qs, qc, rs, rc);
            dist_tile<WQ, WN, VEC, OUT, DMA, true>(a, qs, qc, rs, rc);
            __syncthreads();  // the tile's LDS is read to the end before the next tile's loads
        }
        return;
    } else {
        // XCD-aware order: workgroup w runs on XCD w % 8.  XCD x takes database tiles x, x+8, ...
        // and runs every query block of a tile back to back, so each tile crosses the fabric once
        // and is reused from that XCD's L2 (the grid is padded to a multiple of 8 tiles).
        const uint32_t nqb = a.gather ? 1u : (a.Q + T::TQ - 1) / T::TQ;
        const uint32_t xcd = blockIdx.x % kXcds, seq = blockIdx.x / kXcds;
        const uint32_t qb = seq % nqb;
        const uint32_t tb = (seq / nqb) * kXcds + xcd;
        if (!a.gather && tb * uint32_t(T::TN) >= a.N) return;  // padding workgroup
        // Tile extent.  Flat launches derive it from blockIdx; gather launches take one query and
        // up to 128 rows of its gather list.
        uint32_t qs = qb * T::TQ, rs = tb * T::TN, qc, rc;
        if (a.gather) {
            qs = blockIdx.x / a.gtiles;
            rs = (blockIdx.x % a.gtiles) * uint32_t(T::TN);
            const uint32_t m = min(a.gcount[qs], a.gcap);
            if (rs >= m) return;  // empty tile (uniform)
            qc = 1;
            rc = min(uint32_t(T::TN), m - rs);
        } else {
            qc = min(uint32_t(T::TQ), a.Q - qs);
            rc = min(uint32_t(T::TN), a.N - rs);
        }
        dist_tile<WQ, WN, VEC, OUT, DMA>(a, qs, qc, rs, rc);
    }
}

template <int WQ, int WN, bool VEC, int OUT, bool DMA, bool PLAN = false>
va_status launch_tile(va_context* ctx, const DistArgs& a) {
    using T = Tile<WQ, WN>;
    const uint64_t nqb = (a.Q + T::TQ - 1) / T::TQ;
    const uint64_t ntb = (a.N + T::TN - 1) / T::TN;
    const uint64_t grid = PLAN ? a.plan.grid
                          : a.gather ? uint64_t(a.Q) * a.gtiles : nqb * ((ntb + kXcds - 1) / kXcds) * kXcds;
    if (grid == 0) return VA_OK;
    if (grid > 0x7FFFFFFFull) return fail(ctx, VA_ERR_INVALID_ARG, "distance grid too large (%llu tiles)", (unsigned long long)grid);
    auto kern = &dist_gemm_kernel<WQ, WN, VEC, OUT, DMA, PLAN>;
    const size_t lds_bytes = DMA ? T::DMA_LDS_BYTES : T::LDS_BYTES;
    if (lds_bytes > 65536) {
        VA_CHECK_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_bytes)));
    }
    kern<<<dim3(uint32_t(grid)), dim3(T::NT), lds_bytes, ctx->stream>>>(a);
    VA_CHECK_LAUNCH(ctx);
    return VA_OK;
}

// Direct loads address rows through 32-bit offsets below kDmaMaxBytes: every query row the
// launch can name, and every row of one tile relative to the tile's first row.
template <int WQ, int WN>
bool dma_fits(const DistArgs& a, bool vec) {
    if (!VA_DIST_DMA || !vec || LDS_STRIDE != KC) return false;
    const uint64_t qrows = a.qrow ? a.q_rows : a.Q;
    if (qrows == 0) return false;
    const uint64_t tn = a.plan.pre ? Tile<WQ, WN>::TN : std::min<uint64_t>(Tile<WQ, WN>::TN, a.N);
    return (qrows - 1) * uint64_t(a.ldq) * 4 + uint64_t(a.D) * 4 <= kDmaMaxBytes &&
           (tn - 1) * uint64_t(a.ldx) * 4 + uint64_t(a.D) * 4 <= kDmaMaxBytes;
}

template <int WQ, int WN, int OUT>
va_status launch_shape(va_context* ctx, const DistArgs& a, bool vec) {
    if (a.plan.pre) {
        if constexpr (OUT == OUT_FILTER) {
            if constexpr (LDS_STRIDE == KC)
                if (dma_fits<WQ, WN>(a, vec)) return launch_tile<WQ, WN, true, OUT, true, true>(ctx, a);
            return vec ? launch_tile<WQ, WN, true, OUT, false, true>(ctx, a)
                       : launch_tile<WQ, WN, false, OUT, false, true>(ctx, a);
        }
        return fail(ctx, VA_ERR_INVALID_ARG, "launch_dist: planned launches are filter launches");
    }
    if constexpr (LDS_STRIDE == KC)
        if (dma_fits<WQ, WN>(a, vec)) return launch_tile<WQ, WN, true, OUT, true>(ctx, a);
    return vec ? launch_tile<WQ, WN, true, OUT, false>(ctx, a) : launch_tile<WQ, WN, false, OUT, false>(ctx, a);
}

// ---------------------------------------------------------------------------------------
// Few queries: rows streamed into registers
// ---------------------------------------------------------------------------------------
// A batch of at most 32 queries is bound by reading the rows, and a launch of few tiles by the
// latency of each tile's chain of stages (one stage ahead: 1.4 us per 16 values of a row, 104 us for
// 20,000 x 768).  Here every wave is an independent worker without LDS or barriers: a tile of 32
// rows x 32 queries, both operands loaded straight into registers in chunks of 32 values (whole
// 128-byte lines per row), a ring of R chunks with R - 1 in flight.  (Two query blocks per wave
// spilled; the blocks of a batch past 32 are neighbouring tiles instead, which share the rows
// through L2.)  The values of a key are formed
// in dist_tile's order (32x32x2 MFMA steps over d = 8g + e and 8g + 4 + e, exactly ceil(D / 16)
// stages of 16, the norms as two half chains), so the keys are the same bits.  The distance is a
// template parameter: sixteen copies of its switch would be most of the kernel's code.
// Measured against one-wave GEMM tiles, whole searches, top-10: 20,000 x 768, Q = 1 104 -> 38 us;
// 200,000 x 768, Q = 8 189 -> 186; 500,000 x 768, Q = 1 390 -> 353 (1.5 GB: 4.4 TB/s).
// TAIL: D % 4 != 0 (a lane's four values may run into the next row: cleared past D).
// A launch of at most one wave per SIMD is bound by its waves' own chains: R = 8 there, one wave per
// workgroup so that they spread over the CUs (1,024 x 768, Q = 16: 24.6 -> 21.2 us; a search of 5,000 x 128, Q = 1: 18.4 -> 17.0).
template <int R, bool TAIL, int OUT, int OP>
__global__ __launch_bounds__(256, R > 4 ? 1 : 2) void dist_stream_kernel(DistArgs a) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t D = a.D, nch = (D + 31) / 32, nqb = (a.Q + 31) / 32;
    const uint32_t ntiles = (a.N + 31) / 32 * nqb;
    struct Slot {
        f32x4v x[4], q[4];
    };
    const uint32_t nw = blockDim.x >> 6;
    for (uint32_t tile = blockIdx.x * nw + wave; tile < ntiles; tile += gridDim.x * nw) {
        const uint32_t rt = nqb == 1 ? tile : tile / nqb;
        const uint32_t q0 = (tile - rt * nqb) * 32, qn = min(32u, a.Q - q0);
        const __amdgpu_buffer_rsrc_t qres =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.q + int64_t(q0) * a.ldq), 0,
                                              int((uint64_t(qn - 1) * uint64_t(a.ldq) + D) * 4u), 0x00020000);
        const uint32_t qoff = uint32_t(l32) < qn ? uint32_t(l32 * uint64_t(a.ldq) * 4) : kDmaSkip;
        const uint32_t rs = rt * 32, rc = min(32u, a.N - rs);
        const __amdgpu_buffer_rsrc_t xres =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x + int64_t(rs) * a.ldx), 0,
                                              int((uint64_t(rc - 1) * uint64_t(a.ldx) + D) * 4u), 0x00020000);
        const uint32_t xoff = uint32_t(l32) < rc ? uint32_t(l32 * uint64_t(a.ldx) * 4) : kDmaSkip;
        Slot ring[R];
        auto load = [&](uint32_t c, Slot& s) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t d = 32 * c + 8 * g + 4 * hh;
                const bool in = d < D;
                auto one = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t off) {
                    f32x4v v = __builtin_bit_cast(
                        f32x4v, __builtin_amdgcn_raw_buffer_load_b128(r, in && off != kDmaSkip ? off + 4 * d : kDmaSkip, 0, 0));
                    return v;
                };
                s.x[g] = one(xres, xoff);
                s.q[g] = one(qres, qoff);
            }
        };
        f32x16 acc;
        float qss = 0.0f, xss = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
        auto stage = [&](Slot& s, uint32_t c, int h, bool last) {
#pragma unroll
            for (int g = 2 * h; g < 2 * h + 2; ++g) {
                if (TAIL && last) {
                    const uint32_t d = 32 * c + 8 * g + 4 * hh;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (d + e >= D) {
                            s.x[g][e] = 0.0f;
                            s.q[g][e] = 0.0f;
                        }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) xss = fmaf(s.x[g][e], s.x[g][e], xss);
#pragma unroll
                for (int e = 0; e < 4; ++e) qss = fmaf(s.q[g][e], s.q[g][e], qss);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s.x[g][e], s.q[g][e], acc, 0, 0, 0);
            }
        };
#pragma unroll
        for (int r = 0; r < R - 1; ++r) load(uint32_t(r), ring[r]);
        const uint32_t nfull = (nch - 1) / R * R;  // chunks of the rolled loop: none is the last
        for (uint32_t c = 0; c < nfull; c += R) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                load(c + uint32_t(r + R - 1), ring[(r + R - 1) % R]);  // (past the end: zeros, unused)
                stage(ring[r], c + r, 0, false);
                stage(ring[r], c + r, 1, false);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (nfull + R - 1 < nch) load(nfull + R - 1, ring[R - 1]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t c = nfull + r;
            if (c < nch) {
                stage(ring[r], c, 0, true);
                if (32 * c + 16 < D) stage(ring[r], c, 1, true);
            }
        }
        // lane (l32, hh): query q0 + l32 against rows 8j + 4hh + e in acc[4j + e]
        const float xt = xss + __shfl_xor(xss, 32);
        const float qq = qss + __shfl_xor(qss, 32);
        const uint32_t qi = q0 + uint32_t(l32);
        uint32_t key[16];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                key[4 * j + e] = key_of_float(apply_op(OP, acc[4 * j + e], qq, __shfl(xt, 8 * j + 4 * hh + e)));
        if (uint32_t(l32) >= qn) continue;
        if (OUT == OUT_KEYS) {
            uint32_t* o = a.out_k + int64_t(qi) * a.ldo + rs;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t r = 8 * j + 4 * hh + e;
                    if (r < rc) o[r] = key[4 * j + e];
                }
        } else {
            const uint32_t thr = a.thr[qi];
            uint32_t pass = 0;
#pragma unroll
            for (int v = 0; v < 16; ++v)
                pass |= uint32_t((8u * (v >> 2) + 4u * hh + (v & 3) < rc) & (key[v] <= thr)) << v;
            if (!pass) continue;
            uint32_t pos = atomicAdd(a.cnt + qi, uint32_t(__popc(pass)));
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                if (!((pass >> v) & 1)) continue;
                if (pos < a.cap) {
                    const int64_t o = int64_t(qi) * a.cap + pos;
                    a.cand_key[o] = key[v];
                    a.cand_id[o] = a.id_base + rs + 8 * (v >> 2) + 4 * hh + (v & 3);
                }
                ++pos;
            }
        }
    }
}

// The launches dist_stream_kernel takes: keys or a filter over dense query rows, at most 32 queries
// or so few GEMM tiles that the chip would be mostly idle (past that the GEMM's tiles read the rows
// once for up to 128 queries: 500,000 x 768, Q = 40 595 us on them, 810 streamed; 4,096 x 768 centroids,
// Q = 1,024 86 and 110), every offset within a tile below 2^31.
// Every wave reads its 32 queries again for each tile of rows, which costs a filter pass over many long
// rows more than the GEMM's shared stages and latency: about (Q - 6) per value of a row against a fixed
// 60 to 150 us.  Whole searches, streamed / GEMM, us: 2M x 768, Q = 8 1,457 / 1,399, 16 1,642 / 1,429, 32
// 1,992 / 1,432; 500,000 x 768, Q = 16 454 / 407, 32 542 / 411; 1M x 512, Q = 16 519 / 543, 32 621 / 547;
// 130,000 x 768, Q = 64 271 / 185.  Short rows (2M x 100, Q = 32 316 / 390; 1M x 300, Q = 24 420 / 439) and
// rows the GEMM cannot load as 16-byte pieces (1M x 513, Q = 32 848 / 1,044) are streamed.
constexpr uint32_t kStreamDims = 384;
constexpr uint64_t kStreamWork = 5'200'000'000ull;
bool stream_ok(const va_context* ctx, const DistArgs& a, int wq, int wn, bool vec) {
    if (a.wq || a.wn || a.plan.pre || a.gather || a.qrow || a.ids || (a.out != OUT_KEYS && a.out != OUT_FILTER)) return false;
    if (a.op != OP_L2SQ && a.op != OP_L2 && a.op != OP_COS_DIST && a.op != OP_NEG_DOT) return false;
    if (uint64_t(ceil_div(a.N, 32)) * ceil_div(a.Q, 32) >= (1ull << 31)) return false;
    if (uint64_t(31) * uint64_t(a.ldq) * 4 + uint64_t(a.D) * 4 > kDmaMaxBytes ||
        uint64_t(31) * uint64_t(a.ldx) * 4 + uint64_t(a.D) * 4 > kDmaMaxBytes)
        return false;
    if (vec && a.out == OUT_FILTER && a.Q > 6 && a.D >= kStreamDims &&
        uint64_t(a.N) * a.D >= kStreamWork / (a.Q - 6))
        return false;
    if (a.Q <= 32) return true;
    const uint64_t waves = uint64_t(ceil_div(a.N, 32)) * ceil_div(a.Q, 32);
    return (a.Q <= 64 || waves <= 8ull * uint64_t(ctx->num_cus)) &&
           uint64_t(ceil_div(a.Q, 32 * wq)) * ceil_div(a.N, 128 * wn) < 2ull * uint64_t(ctx->num_cus);
}

template <int OUT, int OP>
void launch_stream_op(va_context* ctx, const DistArgs& a) {
    const uint32_t tiles = ceil_div(a.N, 32) * ceil_div(a.Q, 32);
    const uint32_t grid = std::min((tiles + 3) / 4, 8 * uint32_t(ctx->num_cus));
    if (tiles <= 4 * uint32_t(ctx->num_cus)) {
        if (a.D % 4) dist_stream_kernel<8, true, OUT, OP><<<dim3(tiles), dim3(64), 0, ctx->stream>>>(a);
        else dist_stream_kernel<8, false, OUT, OP><<<dim3(tiles), dim3(64), 0, ctx->stream>>>(a);
    } else if (a.D % 4)
        dist_stream_kernel<4, true, OUT, OP><<<dim3(grid), dim3(256), 0, ctx->stream>>>(a);
    else
        dist_stream_kernel<4, false, OUT, OP><<<dim3(grid), dim3(256), 0, ctx->stream>>>(a);
}
template <int OUT>
va_status launch_stream(va_context* ctx, const DistArgs& a) {
    switch (a.op) {
        case OP_L2SQ: launch_stream_op<OUT, OP_L2SQ>(ctx, a); break;
        case OP_L2: launch_stream_op<OUT, OP_L2>(ctx, a); break;
        case OP_COS_DIST: launch_stream_op<OUT, OP_COS_DIST>(ctx, a); break;
        default: launch_stream_op<OUT, OP_NEG_DOT>(ctx, a);
    }
    VA_CHECK_LAUNCH(ctx);
    return VA_OK;
}

}  // namespace

va_status launch_dist(va_context* ctx, const DistArgs& a) {
    if (a.plan.pre ? a.plan.grid == 0 : (a.Q == 0 || a.N == 0)) return VA_OK;
    const bool vec = (a.D % 4 == 0) && (a.ldq % 4 == 0) && (a.ldx % 4 == 0) &&
                     ((reinterpret_cast<uintptr_t>(a.q) & 15) == 0) && ((reinterpret_cast<uintptr_t>(a.x) & 15) == 0);
    if (a.gather) {
        // rows come from anywhere in the database (64-bit addresses): register-staged loads
        if (a.out != OUT_KEYS || a.plan.pre || a.qrow || a.gtiles == 0 || a.gcap == 0 || !a.gcount)
            return fail(ctx, VA_ERR_INVALID_ARG, "launch_dist: malformed gather launch");
        return vec ? launch_tile<1, 1, true, OUT_KEYS, false>(ctx, a) : launch_tile<1, 1, false, OUT_KEYS, false>(ctx, a);
    }
    const int wq = a.wq ? a.wq : (a.Q <= 32 ? 1 : (a.Q <= 64 ? 2 : 4));
    const int wn = a.wn ? a.wn : 4 / wq;
    if (stream_ok(ctx, a, wq, wn, vec))
        return a.out == OUT_KEYS ? launch_stream<OUT_KEYS>(ctx, a) : launch_stream<OUT_FILTER>(ctx, a);
#define VA_DIST_CASE(W, N, O) \
    if (wq == W && wn == N && a.out == O) return launch_shape<W, N, O>(ctx, a, vec);
    VA_DIST_CASE(1, 4, OUT_VALUES) VA_DIST_CASE(1, 4, OUT_KEYS) VA_DIST_CASE(1, 4, OUT_FILTER)
    VA_DIST_CASE(2, 2, OUT_VALUES) VA_DIST_CASE(2, 2, OUT_KEYS) VA_DIST_CASE(2, 2, OUT_FILTER)
    VA_DIST_CASE(4, 1, OUT_VALUES) VA_DIST_CASE(4, 1, OUT_KEYS) VA_DIST_CASE(4, 1, OUT_FILTER)
    VA_DIST_CASE(1, 4, OUT_ARGMIN) VA_DIST_CASE(2, 2, OUT_ARGMIN) VA_DIST_CASE(4, 1, OUT_ARGMIN)
    // small list-major tiles (one or two waves) for sparse IVF work
    VA_DIST_CASE(1, 1, OUT_FILTER) VA_DIST_CASE(2, 1, OUT_FILTER)
#undef VA_DIST_CASE
    return fail(ctx, VA_ERR_INVALID_ARG, "launch_dist: no %dx%d tile for output mode %d", wq, wn, int(a.out));
}

}  // namespace va
