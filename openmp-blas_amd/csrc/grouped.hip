// Grouped execution: thousands of independent GEMMs and GEMVs in ONE
// persistent kernel launch, captured in a hipGraph.  (The reference has no
// batched API; a caller loops over mtm_helper / mtv_helper.)
//
// Work list: every GEMM is cut into tiles of the class the autotuner chose
// for its (log2 M, log2 N, log2 K) bucket, every GEMV into 64-row chunks;
// items are sorted by estimated cost (longest first).  A fixed grid of
// workgroups (CUs x occupancy) pulls chunks of consecutive items from an
// atomic counter; the last workgroup to finish resets the counters (atomics
// only: no cache-flushing fences, no memset node in the graph).
//
// Every tile class keeps the per-element arithmetic of the standalone kernels
// (plain: sequential k FMAs folded every 128 k; split-BF16: the same MFMA
// slices, product order and 256-k folds; scaled split-FP16: the same line
// exponents, pieces and products; GEMV: the same lane order and butterfly),
// so a grouped result is bitwise the one omb_sgemm / omb_sgemv gives for
// that instance alone -- whatever else is in the batch -- with one
// exception: for K > 512 and few output tiles omb_sgemm may split K into
// coarse blocks of several accumulation blocks each, which rounds
// differently; grouped tiles never split K, so such an instance keeps the
// unsplit fold (same error bound, other bits).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <tuple>
#include <vector>

#include "gemv_row.hpp"
#include "host_util.hpp"
#include "sgemm_wave.hpp"
#include "split_tile.hpp"

namespace omb {
namespace {

struct DGemm {
    int64_t M, N, K;
    const float* A;
    int64_t lda;
    const float* B;
    int64_t ldb;
    float* C;
    int64_t ldc;
    float alpha, beta;
    int* ea;  // scaled FP16 split: exponent of every row of A, every column of B
    int* eb;
};

// Exponent work of the scaled FP16 split: rows start .. start+31 of A (8
// per wavefront) or columns start .. start+63 of B (a lane per column, the
// k range shared by the 4 wavefronts).
constexpr int kExpRows = 32, kExpCols = 64;
struct ExpItem {
    int inst, col;
    int64_t start;
};

struct DGemv {
    int64_t M, N;
    const float* A;
    int64_t lda;
    const float* x;
    float* y;
    float alpha, beta;
};

constexpr int kTileM[NCLS] = {32, 64, 128, 64, 64};
constexpr int kTileN[NCLS] = {32, 64, 64, 64, 1};

struct Item {
    int cls, inst, tm, tn;
};

struct PArgs {
    const Item* items;
    int nitems;
    const DGemm* gemms;
    const DGemv* gemvs;
    unsigned* counters;  // [0] next dynamic chunk, [1] workgroups done
    int chunk;    // consecutive items per chunk
    int nchunks;  // ceil(nitems / chunk)
};

constexpr int NT = 256;
constexpr int kFoldK = 128;  // k per inner accumulation block (as sgemm_f32)

// threadIdx.x through an empty asm, read at the start of every item: index
// math derived from it cannot be hoisted out of the persistent kernel's item
// loop, where it would hold registers for every item type across all items.
__device__ __forceinline__ int item_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// ------------------------------------------------------------ plain tile --
// 128 x 64 tile of C = alpha*A*B + beta*C (all row-major); 256 threads on a
// 16 x 16 grid.  Thread (ty, tx) owns rows g*64 + ty*4 + i (g < 2, i < 4) and
// columns tx*4 + j (j < 4), so every LDS read is one 128-bit access.  Slices of
// 16 k are loaded with 128-bit global loads along the unit-stride index one slice
// ahead and staged through two LDS buffers; LDS fragments for k+1 are read while
// k's FMAs run.  Every element sums k in order and folds the running sum every
// 128 k, as sgemm_f32_kernel does, so the results are the same bits.
template <typename P>
__device__ __forceinline__ float4 load4_guard(P p, int n) {
    if (n == 4) return ld4u(p);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (n > 0) v.x = p[0];
    if (n > 1) v.y = p[1];
    if (n > 2) v.z = p[2];
    return v;
}

__device__ __forceinline__ int clamp4i(int64_t r) { return r <= 0 ? 0 : (r >= 4 ? 4 : (int)r); }

__device__ __forceinline__ void tile_128x64(const DGemm& g, int tm, int tn, float* smem) {
    constexpr int BM = 128, BN = 64, BK = 16, W = 16;  // W: threads along a row of the tile
    constexpr int GR = BM / 64, TMR = 4 * GR, TNR = 4;
    constexpr int kFold = kFoldK / BK;
    constexpr int PA = BM + 4, PB = BN + 4;  // padded LDS rows, 16-byte aligned
    constexpr int LA = BM * BK / 4 / NT, LB = BN * BK / 4 / NT;  // float4 per thread and slice
    static_assert(LA * NT * 4 == BM * BK && LB * NT * 4 == BN * BK, "whole loads");
    // Two LDS buffers of [BK][PA] A and [BK][PB] B: slice k+1 is stored into
    // one while slice k is read from the other (one barrier per slice).
    constexpr int SZ = BK * (PA + PB);
    const int tid = item_tid(), tx = tid % W, ty = tid / W;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int64_t M = g.M, N = g.N, K = g.K;
    gcfloat* const gA = as_global(g.A);
    gcfloat* const gB = as_global(g.B);
    gfloat* const gC = as_global(g.C);

    float4 ra[LA], rb[LB];  // the slice in flight
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {  // A[m][k]: float4 along k
            const int e = tid + i * NT;
            const int row = e >> 2, kq = (e & 3) * 4;
            const int64_t m = m0 + row, k = k0 + kq;
            const int n = m < M ? clamp4i(K - k) : 0;
            ra[i] = load4_guard(gA + (n ? m * g.lda + k : 0), n);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {  // B[k][n]: float4 along n
            const int e = tid + i * NT;
            const int kk = e / (BN / 4), nq = (e % (BN / 4)) * 4;
            const int64_t nn = n0 + nq, k = k0 + kk;
            const int n = k < K ? clamp4i(N - nn) : 0;
            rb[i] = load4_guard(gB + (n ? k * g.ldb + nn : 0), n);
        }
    };
    auto store = [&](int buf) {
        float* As = smem + buf * SZ;
        float* Bs = As + BK * PA;
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int e = tid + i * NT;
            const int row = e >> 2, kq = (e & 3) * 4;
            As[(kq + 0) * PA + row] = ra[i].x;
            As[(kq + 1) * PA + row] = ra[i].y;
            As[(kq + 2) * PA + row] = ra[i].z;
            As[(kq + 3) * PA + row] = ra[i].w;
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int e = tid + i * NT;
            const int kk = e / (BN / 4), nq = (e % (BN / 4)) * 4;
            *reinterpret_cast<float4*>(&Bs[kk * PB + nq]) = rb[i];
        }
    };

    float inner[TMR][TNR], outer[TMR][TNR];
#pragma unroll
    for (int i = 0; i < TMR; ++i)
#pragma unroll
        for (int j = 0; j < TNR; ++j) inner[i][j] = outer[i][j] = 0.f;

    const int64_t nk = ceil_div(K, BK);
    auto compute = [&](int buf, int64_t kt) {
        const float* As = smem + buf * SZ;
        const float* Bs = As + BK * PA;
        float4 fa[2][GR], fb[2];
        auto fragment = [&](int k, int set) {
#pragma unroll
            for (int q = 0; q < GR; ++q)
                fa[set][q] = *reinterpret_cast<const float4*>(&As[k * PA + q * 64 + ty * 4]);
            fb[set] = *reinterpret_cast<const float4*>(&Bs[k * PB + tx * 4]);
        };
        fragment(0, 0);
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            if (k + 1 < BK) fragment(k + 1, (k + 1) & 1);
            const float* av = reinterpret_cast<const float*>(fa[k & 1]);
            const float* bv = reinterpret_cast<const float*>(&fb[k & 1]);
#pragma unroll
            for (int i = 0; i < TMR; ++i)
#pragma unroll
                for (int j = 0; j < TNR; ++j) inner[i][j] = fmaf(av[i], bv[j], inner[i][j]);
        }
        if ((kt + 1) % kFold == 0 || kt + 1 == nk) {
#pragma unroll
            for (int i = 0; i < TMR; ++i)
#pragma unroll
                for (int j = 0; j < TNR; ++j) {
                    outer[i][j] += inner[i][j];
                    inner[i][j] = 0.f;
                }
        }
    };
    // Step kt loads slice kt + 1, computes slice kt from LDS buffer kt % 2 and
    // stores slice kt + 1 into the other buffer.
    load(0);  // also when K = 0 (zeros)
    __syncthreads();  // the previous item is done with LDS
    store(0);
    __syncthreads();
    for (int64_t kt = 0; kt < nk; ++kt) {
        if (kt + 1 < nk) load((kt + 1) * BK);
        compute((int)(kt & 1), kt);
        // The other buffer was last read in step kt - 1, which every thread
        // finished before the barrier that ended it.
        if (kt + 1 < nk) store((int)((kt + 1) & 1));
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TMR; ++i) {
        const int64_t m = m0 + (i / 4) * 64 + ty * 4 + (i % 4);
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TNR; ++j) {
            const int64_t n = n0 + tx * 4 + j;
            if (n < N) {
                gfloat* c = gC + m * g.ldc + n;
                const float v = g.alpha * outer[i][j];
                *c = g.beta != 0.f ? v + g.beta * *c : v;
            }
        }
    }
}

// -------------------------------------------------- wavefront-private tiles --
// One wavefront's 32 x 32 of C = alpha*A*B + beta*C at (m0, n0) (row-major):
// the row and column quads of a lane, as sgemm_wave.hpp lays them out.
typedef wave::WaveSide<32, true, int64_t, gcfloat*> SideA;
typedef wave::WaveSide<32, false, int64_t, gcfloat*> SideB;

// C's rows i0 .. i0 + R - 1 of each lane's four, whole quads at any alignment, the
// reads of C ahead of the writes.
template <int R>
__device__ __forceinline__ void store_quads(const DGemm& g, int64_t m0, int64_t n0, int lane, int i0,
                                            const acc4 (&v)[R]) {
    typedef OMB_GLOBAL f32x4_u gf32x4_u;
    const int rows = (int)std::min<int64_t>(g.M - m0, 32), cols = (int)std::min<int64_t>(g.N - n0, 32);
    const int m = (lane >> 3) * 4 + i0, n = (lane & 7) * 4;
    if (n >= cols) return;
    gfloat* const c = as_global(g.C) + (m0 + m) * g.ldc + n0 + n;
    float4 old[R];
    if (g.beta != 0.f) {
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (m + i < rows && n + 3 < cols) old[i] = ld4u((gcfloat*)(c + i * g.ldc));
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
        if (m + i >= rows) continue;
        f32x4_u x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = g.alpha * v[i][acc_slot(j)];
        if (n + 3 < cols) {
            if (g.beta != 0.f)
                x = f32x4_u{x[0] + g.beta * old[i].x, x[1] + g.beta * old[i].y,
                            x[2] + g.beta * old[i].z, x[3] + g.beta * old[i].w};
            *reinterpret_cast<gf32x4_u*>(c + i * g.ldc) = x;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (n + j < cols) {
                    gfloat* e = c + i * g.ldc + j;
                    *e = g.beta != 0.f ? x[j] + g.beta * *e : x[j];
                }
        }
    }
}

// 64 x 64 as four 32 x 32 quadrants, one per wavefront, each through all of K with
// slices of its own: no barrier in the k loop, and a quadrant past C costs nothing.
// Two slices of loads are in flight; the running sum folds every 128 k, as in
// sgemm_f32_kernel, so the results are the same bits.  Bound by the LDS reads (two
// 128-bit reads per 16 FMAs) and, for few k, by each slice's latency; 4096 GEMMs of
// 16 to 512 took 784 us as 64 x 64 tiles of the whole workgroup, 613 so.
__device__ __forceinline__ void tile_quads(const DGemm& g, int tm, int tn, float* smem) {
    using namespace wave;
    const int tid = item_tid(), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t m0 = (int64_t)tm * 64 + (w >> 1) * 32, n0 = (int64_t)tn * 64 + (w & 1) * 32;
    if (m0 >= g.M || n0 >= g.N) return;
    WaveStage<1, 1>& st = reinterpret_cast<WaveStage<1, 1>*>(smem)[w];
    SideA sa;
    SideB sb;
    sa.init(as_global(g.A), g.lda, m0, g.M, lane);
    sb.init(as_global(g.B), g.ldb, n0, g.N, lane);
    int64_t oa[sa.L], ob[sb.L];
#pragma unroll
    for (int i = 0; i < sa.L; ++i) oa[i] = sa.offset(i);
#pragma unroll
    for (int i = 0; i < sb.L; ++i) ob[i] = sb.offset(i);
    acc4 inner[4][1], outer[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) inner[i][0] = outer[i] = acc4{0.f, 0.f, 0.f, 0.f};
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            outer[i] += inner[i][0];
            inner[i][0] = acc4{0.f, 0.f, 0.f, 0.f};
        }
    };
    const int64_t K = g.K, nfull = full_slices(K, 0, std::max(sa.tail(), sb.tail()));
    float4 va[2][sa.L], vb[2][sb.L];
    auto load = [&](int set, int64_t s) {
        const int64_t k0 = std::min(s, nfull - 1) * BK;
        sa.load(va[set], oa, k0);
        sb.load(vb[set], ob, k0);
    };
    auto store = [&](int set) {
        wave_lds_fence();
        sa.store(st.a, va[set]);
        sb.store(st.b, vb[set]);
        wave_lds_fence();
    };
    int64_t s = 0;
    if (nfull > 0) {
        load(0, 0);
        load(1, 1);
        // whole pairs, with the slice index of the loads clamped to the last one
        for (; s + 1 < nfull; s += 2) {
            pin(inner);
            store(0);
            load(0, s + 2);
            __builtin_amdgcn_sched_barrier(0);
            wave_compute<1, 1>(st, lane, inner);
            store(1);
            load(1, s + 3);
            __builtin_amdgcn_sched_barrier(0);
            wave_compute<1, 1>(st, lane, inner);
            if ((s + 2) % (BLOCK_K / BK) == 0) fold();
        }
        if (s < nfull) {
            store(0);
            wave_compute<1, 1>(st, lane, inner);
            if (++s % (BLOCK_K / BK) == 0) fold();
        }
    }
    for (int64_t k = s * BK; k < K; k += BK) {
        sa.load_guarded(va[0], k, std::min<int64_t>(K, k + BK));
        sb.load_guarded(vb[0], k, std::min<int64_t>(K, k + BK));
        store(0);
        wave_compute<1, 1>(st, lane, inner);
        if ((k + BK) % BLOCK_K == 0) fold();
    }
    if (K % BLOCK_K || K == 0) fold();
    store_quads<4>(g, m0, n0, lane, 0, outer);
}

// 32 x 32 with K divided among the workgroup's wavefronts by 128-k blocks, whose
// sums meet in LDS in block order (the fold, and the bits, of the other tiles).
// For products with a short side and several blocks, whose few tiles would each
// take all of K in one chain.
__device__ __forceinline__ void tile_shared_k(const DGemm& g, int tm, int tn, float* smem) {
    using namespace wave;
    constexpr int W = NT / 64;
    const int tid = item_tid(), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t m0 = (int64_t)tm * 32, n0 = (int64_t)tn * 32, K = g.K;
    WaveStage<1, 1>& st = reinterpret_cast<WaveStage<1, 1>*>(smem)[w];
    acc4* sum = reinterpret_cast<acc4*>(smem);  // [W][4][64], after a round's staging
    SideA sa;
    SideB sb;
    sa.init(as_global(g.A), g.lda, m0, g.M, lane);
    sb.init(as_global(g.B), g.ldb, n0, g.N, lane);
    int64_t oa[sa.L], ob[sb.L];
#pragma unroll
    for (int i = 0; i < sa.L; ++i) oa[i] = sa.offset(i);
#pragma unroll
    for (int i = 0; i < sb.L; ++i) ob[i] = sb.offset(i);
    const int tail = std::max(sa.tail(), sb.tail());
    acc4 outer[1] = {acc4{0.f, 0.f, 0.f, 0.f}};  // row w of each lane's four
    const int64_t nblk = ceil_div(K, (int64_t)BLOCK_K);
    for (int64_t first = 0; first < nblk; first += W) {
        acc4 inner[4][1];
#pragma unroll
        for (int i = 0; i < 4; ++i) inner[i][0] = acc4{0.f, 0.f, 0.f, 0.f};
        const int64_t kb = (first + w) * BLOCK_K, ke = std::min<int64_t>(K, kb + BLOCK_K);
        if (kb < K) {
            const int nfull = full_slices((int)(ke - kb), K - ke, tail);
            float4 va[2][sa.L], vb[2][sb.L];
            auto load = [&](int set, int s) {
                const int64_t k0 = kb + std::min(s, nfull - 1) * BK;
                sa.load(va[set], oa, k0);
                sb.load(vb[set], ob, k0);
            };
            auto store = [&](int set) {
                wave_lds_fence();
                sa.store(st.a, va[set]);
                sb.store(st.b, vb[set]);
                wave_lds_fence();
            };
            int s = 0;
            if (nfull > 0) {
                load(0, 0);
                load(1, 1);
                for (; s + 1 < nfull; s += 2) {
                    pin(inner);
                    store(0);
                    load(0, s + 2);
                    __builtin_amdgcn_sched_barrier(0);
                    wave_compute<1, 1>(st, lane, inner);
                    store(1);
                    load(1, s + 3);
                    __builtin_amdgcn_sched_barrier(0);
                    wave_compute<1, 1>(st, lane, inner);
                }
                if (s < nfull) {
                    store(0);
                    wave_compute<1, 1>(st, lane, inner);
                    ++s;
                }
            }
            for (int64_t k = kb + s * BK; k < ke; k += BK) {
                sa.load_guarded(va[0], k, std::min<int64_t>(ke, k + BK));
                sb.load_guarded(vb[0], k, std::min<int64_t>(ke, k + BK));
                store(0);
                wave_compute<1, 1>(st, lane, inner);
            }
        }
        const int in_round = (int)std::min<int64_t>(W, nblk - first);
        __syncthreads();  // the staging buffers are read
        if (w < in_round) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[(w * 4 + i) * 64 + lane] = inner[i][0];
        }
        __syncthreads();
        for (int b = 0; b < in_round; ++b) outer[0] += sum[(b * 4 + w) * 64 + lane];
        __syncthreads();  // before the next round's staging
    }
    store_quads<1>(g, m0, n0, lane, w, outer);
}

// ------------------------------------------------------------ split tile --
// 64x64 tile on the MFMA cores of a row-major A and B (split_tile.hpp): the BF16
// pieces, or (F16) the FP16 pieces of every element scaled by its row's (A) or
// column's (B) exponent, with the sums scaled back when stored.
template <int NPROD, bool F16>
__device__ __forceinline__ void tile_split(const DGemm& g, int tm, int tn, float* smem) {
    using namespace split;
    const int tid = item_tid(), wave = tid >> 6;
    const int64_t m0 = (int64_t)tm * kLines, n0 = (int64_t)tn * kLines;
    Quad<true, gcfloat*> qa;
    Quad<false, gcfloat*> qb;
    qa.init(as_global(g.A), g.lda, m0, g.M, tid);
    qb.init(as_global(g.B), g.ldb, n0, g.N, tid);
    const int rows = (int)std::min<int64_t>(g.M - m0, kLines);
    const int cols = (int)std::min<int64_t>(g.N - n0, kLines);
    gcint* const em = F16 ? as_global(static_cast<const int*>(g.ea)) + m0 : nullptr;
    gcint* const en = F16 ? as_global(static_cast<const int*>(g.eb)) + n0 : nullptr;
    const int ea = F16 ? em[std::min(qa.line, rows - 1)] : 0;
    const int eb = F16 ? en[std::min(qb.line, cols - 1)] : 0;
    float out[16];
    tile_sums<NPROD, F16, 1>(qa, qb, ea, eb, g.K, 0, tid,
                             reinterpret_cast<Staged<NPROD, F16>*>(smem), nullptr, out);
    store_sums(out, 0, wave >> 1, wave & 1, tid & 63, as_global(g.C) + m0 * g.ldc + n0, g.ldc, rows,
               cols, g.alpha, g.beta, em, en);
}

// --------------------------------------------------- scaled FP16 split --
// Line exponents e = 14 - ilogb(max |x|) (0 for a zero, infinite or NaN
// line), one per row of A and column of B.  The maximum is taken over the
// bits of |x| (unsigned order is the numeric order for non-negative floats;
// NaN's bits exceed infinity's) and is order-free, so the exponents are the
// ones omb_sgemm's maxima passes give.
__global__ __launch_bounds__(NT) void grouped_exps_kernel(const ExpItem* __restrict__ items,
                                                          const DGemm* __restrict__ gemms) {
    __shared__ unsigned red[NT];
    const ExpItem w = items[blockIdx.x];
    const DGemm& g = gemms[w.inst];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int RW = kExpRows / (NT / 64);  // rows per wavefront
    if (w.col == 0) {
        const int64_t m0 = w.start + wave * RW;
        unsigned mx[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) mx[r] = 0;
        for (int64_t k = lane; k < g.K; k += 64) {
#pragma unroll
            for (int r = 0; r < RW; ++r)  // RW independent loads in flight
                if (m0 + r < g.M) {
                    const unsigned b = __float_as_uint(g.A[(m0 + r) * g.lda + k]) & 0x7fffffffu;
                    mx[r] = b > mx[r] ? b : mx[r];
                }
        }
#pragma unroll
        for (int r = 0; r < RW; ++r) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const unsigned o = (unsigned)__shfl_xor((int)mx[r], off);
                mx[r] = o > mx[r] ? o : mx[r];
            }
            if (lane == r && m0 + r < g.M) g.ea[m0 + r] = split::line_exp(__uint_as_float(mx[r]));
        }
    } else {
        const int64_t n = w.start + lane;
        unsigned mx = 0;
        if (n < g.N) {
#pragma unroll 8
            for (int64_t k = wave; k < g.K; k += NT / 64) {
                const unsigned b = __float_as_uint(g.B[k * g.ldb + n]) & 0x7fffffffu;
                mx = b > mx ? b : mx;
            }
        }
        red[threadIdx.x] = mx;
        __syncthreads();
        if (wave == 0 && n < g.N) {
#pragma unroll
            for (int q = 1; q < NT / 64; ++q) mx = red[q * 64 + lane] > mx ? red[q * 64 + lane] : mx;
            g.eb[n] = split::line_exp(__uint_as_float(mx));
        }
    }
}

// ------------------------------------------------------------- GEMV item --
__device__ __forceinline__ void gemv_item(const DGemv& v, int chunk) {
    const int tid = item_tid();
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Wavefront w takes rows chunk*64 + 16w .. +15, as many at a time as keep 16
    // loads per lane in flight (16 rows x 1 load, 8 x 2, 4 x 4) with no load past a
    // short row, and with the non-temporal hint: bound by HBM, whose rate the hint
    // raises from 6.3 to 6.8 TB/s for rows of 4096, if the loads of a row come
    // together so that lines at their borders are read once.  4096 GEMVs of 64 to
    // 4096: 2622 us as 16 x 1 without the hint, 2599 with it, 2460 so (6.3 TB/s).
    const int64_t r0 = (int64_t)chunk * 64 + wave * 16;
    if (r0 >= v.M) return;
    const int nr = (int)(v.M - r0 < 16 ? v.M - r0 : 16);
    auto rows = [&](auto rows_at_once, auto loads) {
        constexpr int R = decltype(rows_at_once)::value, U = decltype(loads)::value;
        for (int q = 0; q < nr; q += R)
            gemv_rows_wave<R, U, true, true, true, true>(
                r0 + q, std::min(nr - q, R), v.N, v.alpha, as_global(v.A), v.lda, as_global(v.x),
                v.beta, as_global(v.y), lane);
    };
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, 4> I4;
    if (v.N < 4 * 65) rows(std::integral_constant<int, 16>{}, I1{});
    else if (v.N < 4 * 129) rows(std::integral_constant<int, 8>{}, I2{});
    else if (v.N < kGemvOff32Cols) rows(I4{}, I4{});
    else
        gemv_rows_wave<16, 1, false>(r0, nr, v.N, v.alpha, as_global(v.A), v.lda, as_global(v.x), v.beta,
                                     as_global(v.y), lane);
}

// ------------------------------------------------------- persistent kernel --
// LDS: the largest plain class footprint (128x64: two buffers of
// 16 x (132 + 68) floats); the split tiles use at most 24 KB.
constexpr int kSmemFloats = 2 * (16 * (128 + 4) + 16 * (64 + 4)) + 16;

// One build per kind of GEMM item, so that none holds registers for another's
// (with all in one, the pipelined split tiles cost the plain plan of 4096 GEMMs
// 860 us instead of 783).  All but KBIG are bounded to 4 workgroups per CU (at
// most 128 VGPRs): the plain plan of 4096 GEMMs and 4096 GEMVs measured 3.48 ms
// so, against 3.55-3.63 ms for builds of 129 and 165 VGPRs (3 per CU).  KBIG (128x64
// tiles too) is bounded to 2 and runs 3 (154 VGPRs).
enum Kind { KPLAIN, KBIG, KSPLIT6, KSPLIT3, KSPLIT16, NKIND };

template <int KIND>
__global__ __launch_bounds__(NT, KIND == KBIG ? 2 : 4) void grouped_kernel(PArgs p) {
    __shared__ __attribute__((aligned(16))) float smem[kSmemFloats];
    __shared__ int s_chunk;
    // Chunks of consecutive (cost-sorted) items: workgroup b starts with
    // chunk b, then takes chunks gridDim.x, gridDim.x + 1, ... from one
    // device-scope counter.  Such atomics on one address serialize (about
    // 70 ns each measured here), so one ticket per chunk instead of one per
    // item keeps the counter off the critical path.
    int c = blockIdx.x;
    for (;;) {
        if (c >= p.nchunks) break;
        const int beg = c * p.chunk, end = min(beg + p.chunk, p.nitems);
        for (int it = beg; it < end; ++it) {
            __syncthreads();  // the previous item is done with LDS
            Item w = p.items[it];
            w.cls = __builtin_amdgcn_readfirstlane(w.cls);
            w.inst = __builtin_amdgcn_readfirstlane(w.inst);
            w.tm = __builtin_amdgcn_readfirstlane(w.tm);
            w.tn = __builtin_amdgcn_readfirstlane(w.tn);
            switch (w.cls) {
                case C32:
                    if constexpr (KIND <= KBIG)
                        tile_shared_k(p.gemms[w.inst], w.tm, w.tn, smem);
                    break;
                case C64:
                    if constexpr (KIND <= KBIG)
                        tile_quads(p.gemms[w.inst], w.tm, w.tn, smem);
                    break;
                case C128x64:
                    if constexpr (KIND == KBIG)
                        tile_128x64(p.gemms[w.inst], w.tm, w.tn, smem);
                    break;
                case CSPLIT:
                    if constexpr (KIND >= KSPLIT6)
                        tile_split<KIND == KSPLIT6 ? 6 : 3, KIND == KSPLIT16>(p.gemms[w.inst], w.tm,
                                                                             w.tn, smem);
                    break;
                case CGEMV: gemv_item(p.gemvs[w.inst], w.tm); break;
                default: break;
            }
        }
        __syncthreads();  // every thread has read s_chunk for this chunk
        if (threadIdx.x == 0) s_chunk = (int)gridDim.x + (int)atomicAdd(&p.counters[0], 1u);
        __syncthreads();
        // uniform across the workgroup: keep it (and the descriptors) scalar
        c = __builtin_amdgcn_readfirstlane(s_chunk);
    }
    if (threadIdx.x == 0 && atomicAdd(&p.counters[1], 1u) == gridDim.x - 1) {
        atomicExch(&p.counters[0], 0u);
        atomicExch(&p.counters[1], 0u);
    }
}

typedef void (*GroupedKernel)(PArgs);
GroupedKernel grouped_kernel_of(Kind k) {
    switch (k) {
        case KBIG: return grouped_kernel<KBIG>;
        case KSPLIT6: return grouped_kernel<KSPLIT6>;
        case KSPLIT3: return grouped_kernel<KSPLIT3>;
        case KSPLIT16: return grouped_kernel<KSPLIT16>;
        default: return grouped_kernel<KPLAIN>;
    }
}
Kind kind_of(int mode, bool big) {
    return mode == OMB_MODE_SPLIT_FP16      ? KSPLIT16
           : mode == OMB_MODE_SPLIT_BF16_P3 ? KSPLIT3
           : mode == OMB_MODE_SPLIT_BF16    ? KSPLIT6
           : big                            ? KBIG
                                            : KPLAIN;
}

// ---------------------------------------------------------- tuning table --
using Key = TuneKey;
std::mutex g_tune_mu;
std::map<Key, int>& tune_table() {
    static auto* t = new std::map<Key, int>();
    return *t;
}

int lg(int64_t x) {
    int b = 0;
    while (x > 1) {
        x >>= 1;
        ++b;
    }
    return b;
}

Key key_of(int mode, const omb_gemm_desc& d) { return Key{mode, lg(d.M), lg(d.N), lg(d.K)}; }

// Class without a tuning entry: split mode has one class; plain takes 64x64, or
// 32x32 with K shared by the wavefronts when the smaller output dimension is under
// 48 and K has three accumulation blocks or more (4096 GEMMs: 621 us so, 648 with
// every short side in 32x32, 613 with none, 684 with every such K).  (The
// 128x64 class needs the larger-register kernel, 3 workgroups per CU instead
// of 4, which slows every other item of a mixed plan, so it is used only when a
// loaded tuning table names it.)
int default_class(int mode, const omb_gemm_desc& d) {
    if (mode != OMB_MODE_PLAIN_F32) return CSPLIT;
    return d.K > 2 * kFoldK && std::min(d.M, d.N) < 48 ? C32 : C64;
}

// The table's class for the bucket, if it computes this mode (the loader
// accepts only such entries), else the default.
int choose_class(int mode, const omb_gemm_desc& d) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    auto it = tune_table().find(key_of(mode, d));
    return it != tune_table().end() && class_serves_mode(it->second, mode)
               ? it->second
               : default_class(mode, d);
}

}  // namespace
}  // namespace omb

// ------------------------------------------------------------------ plans --
struct omb_group_plan {
    int dev = 0;
    int mode = 0;
    bool big = false;
    int grid = 0;
    int nitems = 0;
    int chunk = 1;
    omb::DGemm* d_gemms = nullptr;
    omb::DGemv* d_gemvs = nullptr;
    omb::Item* d_items = nullptr;
    unsigned* d_counters = nullptr;
    int nexp = 0;                      // scaled FP16 split: exponent work items
    omb::ExpItem* d_exp_items = nullptr;
    int* d_exps = nullptr;             // every GEMM's row and column exponents
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::string text;
};

namespace omb {
namespace {

omb_status validate(const omb_gemm_desc* gemms, int32_t n_gemm, const omb_gemv_desc* gemvs,
                    int32_t n_gemv) {
    if (n_gemm < 0 || n_gemv < 0 || (n_gemm > 0 && !gemms) || (n_gemv > 0 && !gemvs)) {
        set_error("group plan: bad descriptor array");
        return OMB_EINVAL;
    }
    for (int i = 0; i < n_gemm; ++i) {
        const omb_gemm_desc& d = gemms[i];
        const bool empty = d.M == 0 || d.N == 0;
        if (d.M < 0 || d.N < 0 || d.K < 0 || (!empty && (!d.C || d.ldc < d.N)) ||
            (!empty && d.K > 0 && (!d.A || !d.B || d.lda < d.K || d.ldb < d.N))) {
            set_error("group plan: invalid GEMM descriptor " + std::to_string(i));
            return OMB_EINVAL;
        }
    }
    for (int i = 0; i < n_gemv; ++i) {
        const omb_gemv_desc& d = gemvs[i];
        if (d.M < 0 || d.N < 0 || (d.M > 0 && !d.y) ||
            (d.M > 0 && d.N > 0 && (!d.A || !d.x || d.lda < d.N))) {
            set_error("group plan: invalid GEMV descriptor " + std::to_string(i));
            return OMB_EINVAL;
        }
    }
    return OMB_OK;
}

// Estimated seconds one workgroup spends on an item (for the longest-first
// order): per-workgroup rates -- 32x32 16 GFLOP/s, 64x64 40, 128x64 59, split
// 64x64 54 (FP32-equivalent), GEMV 8 GB/s -- plus about 2 us of fixed cost per item.
// GEMM items count a quarter, so that most follow the GEMV items: the two kinds
// side by side are slower than one after the other (4096 GEMMs alone 613 us, 4096
// GEMVs alone 2608; mixed by equal weights 3356, GEMMs first 3212, GEMVs first 3187,
// at a quarter 3180; 300 of each 314, 329, 321, 314).
constexpr double kGemmOrder = 0.25;
double item_cost(const Item& it, const std::vector<DGemm>& g, const std::vector<DGemv>& v) {
    constexpr double kFixed = 2.0e-6;
    if (it.cls == CGEMV) return kFixed + 64.0 * (double)v[it.inst].N * 4.0 / 8.0e9;
    static const double rate[NCLS] = {16e9, 40e9, 59e9, 54e9, 0.0};
    return kGemmOrder * (kFixed + 2.0 * kTileM[it.cls] * kTileN[it.cls] *
                                      (double)std::max<int64_t>(g[it.inst].K, 1) / rate[it.cls]);
}

template <typename T>
omb_status upload(T** dst, const std::vector<T>& src) {
    *dst = nullptr;
    if (src.empty()) return OMB_OK;
    OMB_HIP_TRY(hipMalloc(reinterpret_cast<void**>(dst), src.size() * sizeof(T)));
    OMB_HIP_TRY(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    return OMB_OK;
}

void free_plan(omb_group_plan* p) {
    if (!p) return;
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    if (p->d_gemms) (void)hipFree(p->d_gemms);
    if (p->d_gemvs) (void)hipFree(p->d_gemvs);
    if (p->d_items) (void)hipFree(p->d_items);
    if (p->d_counters) (void)hipFree(p->d_counters);
    if (p->d_exp_items) (void)hipFree(p->d_exp_items);
    if (p->d_exps) (void)hipFree(p->d_exps);
    delete p;
}

omb_status launch_plan(omb_group_plan* p, hipStream_t s) {
    if (p->nitems == 0) return OMB_OK;
    if (p->nexp > 0) {  // exponents first (same stream: the tiles read them)
        hipLaunchKernelGGL(grouped_exps_kernel, dim3(p->nexp), dim3(NT), 0, s, p->d_exp_items,
                           p->d_gemms);
        OMB_HIP_TRY(hipGetLastError());
    }
    PArgs a{p->d_items, p->nitems, p->d_gemms, p->d_gemvs, p->d_counters, p->chunk,
            (int)ceil_div(p->nitems, p->chunk)};
    hipLaunchKernelGGL(grouped_kernel_of(kind_of(p->mode, p->big)), dim3(p->grid), dim3(NT), 0, s, a);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

// Build a plan; force_cls >= 0 puts every GEMM in that class (autotuner).
omb_status build_plan(const omb_gemm_desc* gemms, int32_t n_gemm, const omb_gemv_desc* gemvs,
                      int32_t n_gemv, int32_t mode, int force_cls, bool capture,
                      omb_group_plan** out) {
    *out = nullptr;
    if (mode != OMB_MODE_PLAIN_F32 && mode != OMB_MODE_SPLIT_BF16 &&
        mode != OMB_MODE_SPLIT_BF16_P3 && mode != OMB_MODE_SPLIT_FP16) {
        set_error("group plan: unknown mode " + std::to_string(mode));
        return OMB_EINVAL;
    }
    OMB_TRY(validate(gemms, n_gemm, gemvs, n_gemv));
    auto* p = new omb_group_plan();
    p->mode = mode;
    std::vector<DGemm> g(n_gemm);
    std::vector<DGemv> v(n_gemv);
    std::vector<Item> items;
    int per_cls[NCLS] = {0, 0, 0, 0, 0};
    std::map<std::string, int> chosen;
    for (int i = 0; i < n_gemm; ++i) {
        const omb_gemm_desc& d = gemms[i];
        g[i] = DGemm{d.M, d.N, d.K, d.A, d.lda, d.B, d.ldb, d.C, d.ldc, d.alpha, d.beta,
                     nullptr, nullptr};
        if (d.M == 0 || d.N == 0) continue;
        const int c = force_cls >= 0 ? force_cls : choose_class(mode, d);
        const int64_t tmn = ceil_div(d.M, kTileM[c]), tnn = ceil_div(d.N, kTileN[c]);
        if (tmn > 0x7fffffff || tnn > 0x7fffffff || (int64_t)items.size() + tmn * tnn > 0x7fffffff) {
            free_plan(p);
            set_error("group plan: too many tiles");
            return OMB_EUNSUPPORTED;
        }
        for (int64_t a = 0; a < tmn; ++a)
            for (int64_t b = 0; b < tnn; ++b) items.push_back(Item{c, i, (int)a, (int)b});
        per_cls[c] += (int)(tmn * tnn);
        if (c == C128x64) p->big = true;
        const Key k = key_of(mode, d);
        chosen["gemm:" + std::to_string(1 << k.bm) + "x" + std::to_string(1 << k.bn) + "x" +
               std::to_string(1 << k.bk) + "=" + kClsName[c]] += 1;
    }
    for (int i = 0; i < n_gemv; ++i) {
        const omb_gemv_desc& d = gemvs[i];
        v[i] = DGemv{d.M, d.N, d.A, d.lda, d.x, d.y, d.alpha, d.beta};
        for (int64_t c = 0; c < ceil_div(d.M, 64); ++c) items.push_back(Item{CGEMV, i, (int)c, 0});
        per_cls[CGEMV] += (int)ceil_div(d.M, 64);
    }
    std::vector<double> cost(items.size());
    for (size_t i = 0; i < items.size(); ++i) cost[i] = item_cost(items[i], g, v);
    std::vector<size_t> order(items.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return cost[a] > cost[b]; });
    std::vector<Item> sorted(items.size());
    for (size_t i = 0; i < order.size(); ++i) sorted[i] = items[order[i]];
    p->nitems = (int)sorted.size();

    omb_status st = OMB_OK;
    if (mode == OMB_MODE_SPLIT_FP16) {
        // one exponent per row of A and column of B, in a plan-owned buffer
        std::vector<ExpItem> ex;
        int64_t lines = 0;
        for (int i = 0; i < n_gemm; ++i)
            if (g[i].M > 0 && g[i].N > 0) lines += g[i].M + g[i].N;
        if (lines > 0 && hipMalloc(&p->d_exps, lines * sizeof(int)) != hipSuccess) {
            (void)hipGetLastError();
            free_plan(p);
            set_error("group plan: exponent allocation failed");
            return OMB_ENOMEM;
        }
        int64_t off = 0;
        for (int i = 0; i < n_gemm; ++i) {
            if (g[i].M == 0 || g[i].N == 0) continue;
            g[i].ea = p->d_exps + off;
            g[i].eb = p->d_exps + off + g[i].M;
            off += g[i].M + g[i].N;
            for (int64_t r = 0; r < g[i].M; r += kExpRows) ex.push_back(ExpItem{i, 0, r});
            for (int64_t c = 0; c < g[i].N; c += kExpCols) ex.push_back(ExpItem{i, 1, c});
        }
        if (ex.size() > 0x7fffffff) {
            free_plan(p);
            set_error("group plan: too many exponent items");
            return OMB_EUNSUPPORTED;
        }
        p->nexp = (int)ex.size();
        if ((st = upload(&p->d_exp_items, ex)) != OMB_OK) {
            free_plan(p);
            return st;
        }
    }
    if ((st = upload(&p->d_gemms, g)) != OMB_OK || (st = upload(&p->d_gemvs, v)) != OMB_OK ||
        (st = upload(&p->d_items, sorted)) != OMB_OK) {
        free_plan(p);
        return st;
    }
    if (hipMalloc(&p->d_counters, 2 * sizeof(unsigned)) != hipSuccess ||
        hipMemset(p->d_counters, 0, 2 * sizeof(unsigned)) != hipSuccess) {
        (void)hipGetLastError();
        free_plan(p);
        set_error("group plan: counter allocation failed");
        return OMB_ENOMEM;
    }
    int dev = 0, cus = 0, per_cu = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
        free_plan(p);
        set_error("group plan: device query failed");
        return OMB_EDEVICE;
    }
    cus = prop.multiProcessorCount;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, grouped_kernel_of(kind_of(p->mode, p->big)), NT, 0);
    if (e != hipSuccess || per_cu < 1) per_cu = 1;
    p->dev = dev;
    p->grid = std::max(1, std::min(p->nitems, cus * per_cu));
    // up to 4 items per chunk (about 8 chunks per workgroup at most): 4x
    // fewer tickets; longer chunks of the cost-sorted list measured slower
    // on mixed GEMM + GEMV plans
    p->chunk = std::max(1, std::min(4, p->nitems / (8 * p->grid)));

    if (capture && p->nitems > 0) {
        hipStream_t cs = nullptr;
        if (hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) {
            free_plan(p);
            set_error("group plan: stream creation failed");
            return OMB_EDEVICE;
        }
        bool ok = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) == hipSuccess;
        ok = ok && launch_plan(p, cs) == OMB_OK;
        ok = hipStreamEndCapture(cs, &p->graph) == hipSuccess && ok;
        ok = ok && hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0) == hipSuccess;
        (void)hipStreamDestroy(cs);
        if (!ok) {
            (void)hipGetLastError();
            free_plan(p);
            set_error("group plan: graph capture failed");
            return OMB_EDEVICE;
        }
    }
    std::ostringstream os;
    os << "items=" << p->nitems << " grid=" << p->grid << " chunk=" << p->chunk
       << " kernel=" << (p->big ? "big" : "lite")
       << " mode=" << mode;
    for (int c = 0; c < NCLS; ++c)
        if (per_cls[c]) os << " " << kClsName[c] << "=" << per_cls[c];
    for (auto& kv : chosen) os << " " << kv.first << "(" << kv.second << ")";
    p->text = os.str();
    *out = p;
    return OMB_OK;
}

}  // namespace
}  // namespace omb

using namespace omb;

extern "C" omb_status omb_group_plan_create(const omb_gemm_desc* gemms, int32_t n_gemm,
                                            const omb_gemv_desc* gemvs, int32_t n_gemv,
                                            int32_t mode, omb_stream_t stream,
                                            omb_group_plan** plan) {
    clear_error();
    (void)stream;  // the graph is captured on a private stream and replayed on any
    if (!plan) {
        set_error("omb_group_plan_create: null plan pointer");
        return OMB_EINVAL;
    }
    return build_plan(gemms, n_gemm, gemvs, n_gemv, mode, -1, true, plan);
}

extern "C" omb_status omb_group_plan_launch(omb_group_plan* plan, omb_stream_t stream) {
    clear_error();
    if (!plan) {
        set_error("omb_group_plan_launch: null plan");
        return OMB_EINVAL;
    }
    if (plan->nitems == 0) return OMB_OK;
    OMB_HIP_TRY(hipGraphLaunch(plan->exec, (hipStream_t)stream));
    return OMB_OK;
}

extern "C" omb_status omb_group_plan_launch_direct(omb_group_plan* plan, omb_stream_t stream) {
    clear_error();
    if (!plan) {
        set_error("omb_group_plan_launch_direct: null plan");
        return OMB_EINVAL;
    }
    return launch_plan(plan, (hipStream_t)stream);
}

extern "C" omb_status omb_group_plan_describe(const omb_group_plan* plan, char* buf, size_t len) {
    clear_error();
    if (!plan || !buf || len == 0) {
        set_error("omb_group_plan_describe: invalid argument");
        return OMB_EINVAL;
    }
    std::snprintf(buf, len, "%s", plan->text.c_str());
    return OMB_OK;
}

extern "C" omb_status omb_group_plan_destroy(omb_group_plan* plan) {
    clear_error();
    free_plan(plan);
    return OMB_OK;
}

// ---------------------------------------------------------------- tuning --
namespace omb {
namespace {

__global__ void tune_fill(float* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        p[i] = rng_uniform(0x5eedULL, (uint64_t)i);
}

// Time `reps` direct launches of a plan that puts `batch` copies of the
// shape in class `cls`; returns milliseconds per launch.
omb_status time_class(int mode, int64_t M, int64_t N, int64_t K, int cls, int batch, float* A,
                      float* B, float* C, hipStream_t s, float* ms) {
    std::vector<omb_gemm_desc> d(batch);
    for (int i = 0; i < batch; ++i)
        d[i] = omb_gemm_desc{M, N, K, A, K, B, N, C + (int64_t)i * M * N, N, 1.f, 0.f};
    omb_group_plan* p = nullptr;
    OMB_TRY(build_plan(d.data(), batch, nullptr, 0, mode, cls, false, &p));
    hipEvent_t e0, e1;
    omb_status st = OMB_OK;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        free_plan(p);
        set_error("autotune: event creation failed");
        return OMB_EDEVICE;
    }
    for (int w = 0; w < 2 && st == OMB_OK; ++w) st = launch_plan(p, s);
    const int reps = 5;
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < reps && st == OMB_OK; ++r) st = launch_plan(p, s);
    (void)hipEventRecord(e1, s);
    if (st == OMB_OK && hipEventSynchronize(e1) == hipSuccess) {
        float t = 0.f;
        (void)hipEventElapsedTime(&t, e0, e1);
        *ms = t / reps;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    free_plan(p);
    return st;
}

}  // namespace
}  // namespace omb

extern "C" omb_status omb_autotune_group(const omb_gemm_desc* gemms, int32_t n_gemm, int32_t mode,
                                         const char* table_path, omb_stream_t stream) {
    clear_error();
    OMB_TRY(validate(gemms, n_gemm, nullptr, 0));
    if (mode != OMB_MODE_PLAIN_F32 && mode != OMB_MODE_SPLIT_BF16 &&
        mode != OMB_MODE_SPLIT_BF16_P3 && mode != OMB_MODE_SPLIT_FP16) {
        set_error("omb_autotune_group: unknown mode");
        return OMB_EINVAL;
    }
    hipStream_t s = (hipStream_t)stream;
    // bucket -> shapes present (the median M*N*K shape represents the bucket)
    std::map<Key, std::vector<omb_gemm_desc>> buckets;
    for (int i = 0; i < n_gemm; ++i)
        if (gemms[i].M > 0 && gemms[i].N > 0) buckets[key_of(mode, gemms[i])].push_back(gemms[i]);
    const int batch = 64;
    // 128x64 is not a candidate: timed alone it can win a bucket, but it
    // needs the larger-register kernel (3 workgroups per CU instead of 4),
    // which slows every other item of the plan (see default_class); a
    // table loaded with omb_autotune_load may still name it.
    const std::vector<int> cands = mode == OMB_MODE_PLAIN_F32 ? std::vector<int>{C32, C64}
                                                              : std::vector<int>{CSPLIT};
    int64_t maxM = 1, maxN = 1, maxK = 1;
    for (auto& kv : buckets)
        for (auto& d : kv.second) {
            maxM = std::max(maxM, d.M);
            maxN = std::max(maxN, d.N);
            maxK = std::max(maxK, d.K);
        }
    float *A = nullptr, *B = nullptr, *C = nullptr;
    if (cands.size() > 1 && !buckets.empty()) {
        if (hipMalloc(&A, maxM * maxK * sizeof(float)) != hipSuccess ||
            hipMalloc(&B, maxK * maxN * sizeof(float)) != hipSuccess ||
            hipMalloc(&C, (size_t)batch * maxM * maxN * sizeof(float)) != hipSuccess) {
            (void)hipGetLastError();
            if (A) (void)hipFree(A);
            if (B) (void)hipFree(B);
            set_error("omb_autotune_group: scratch allocation failed");
            return OMB_ENOMEM;
        }
        hipLaunchKernelGGL(tune_fill, dim3(1024), dim3(256), 0, s, A, maxM * maxK);
        hipLaunchKernelGGL(tune_fill, dim3(1024), dim3(256), 0, s, B, maxK * maxN);
    }
    omb_status st = OMB_OK;
    std::map<Key, int> result;
    for (auto& kv : buckets) {
        if (cands.size() == 1) {
            result[kv.first] = cands[0];
            continue;
        }
        auto shapes = kv.second;
        std::sort(shapes.begin(), shapes.end(), [](const omb_gemm_desc& a, const omb_gemm_desc& b) {
            return a.M * a.N * a.K < b.M * b.N * b.K;
        });
        const omb_gemm_desc rep = shapes[shapes.size() / 2];
        int best = cands[0];
        float best_ms = 1e30f;
        for (int c : cands) {
            float ms = 1e30f;
            st = time_class(mode, rep.M, rep.N, rep.K, c, batch, A, B, C, s, &ms);
            if (st != OMB_OK) break;
            if (ms < best_ms) {
                best_ms = ms;
                best = c;
            }
        }
        if (st != OMB_OK) break;
        result[kv.first] = best;
    }
    if (A) (void)hipFree(A);
    if (B) (void)hipFree(B);
    if (C) (void)hipFree(C);
    if (st != OMB_OK) return st;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        for (auto& kv : result) tune_table()[kv.first] = kv.second;
    }
    if (table_path) {
        std::ofstream f(table_path);
        if (!f) {
            set_error(std::string("omb_autotune_group: cannot write ") + table_path);
            return OMB_EINVAL;
        }
        f << "# mode log2M log2N log2K class\n";
        std::lock_guard<std::mutex> lock(g_tune_mu);
        for (auto& kv : tune_table())
            f << kv.first.mode << " " << kv.first.bm << " " << kv.first.bn << " " << kv.first.bk
              << " " << kClsName[kv.second] << "\n";
    }
    return OMB_OK;
}

extern "C" omb_status omb_autotune_load(const char* table_path) {
    clear_error();
    if (!table_path) {
        set_error("omb_autotune_load: null path");
        return OMB_EINVAL;
    }
    std::ifstream f(table_path);
    if (!f) {
        set_error(std::string("omb_autotune_load: cannot read ") + table_path);
        return OMB_EINVAL;
    }
    std::map<Key, int> loaded;
    std::string err;
    if (!parse_tune_table(f, &loaded, &err)) {
        set_error("omb_autotune_load: " + err);
        return OMB_EINVAL;
    }
    std::lock_guard<std::mutex> lock(g_tune_mu);
    for (auto& kv : loaded) tune_table()[kv.first] = kv.second;
    return OMB_OK;
}

// ---------------------------------------------------------- request batches --
// A grouped launch without a plan object, for the serving loop: the
// descriptors and the cost-sorted item list are built on the host into a
// pinned staging block, copied to the batch's device block on the launch
// stream, and the lite persistent kernel runs them.  Results are bitwise
// those of the grouped plans (and so of the direct calls, see above).  The
// staging block is reused only after the previous launch from it has
// completed, which the caller guarantees (one batch per slot at a time).
namespace omb {

struct GroupBatch {
    char* dev = nullptr;
    char* host = nullptr;
    unsigned* counters = nullptr;
    size_t bytes = 0;
};

namespace {
constexpr int kBatchMaxGemms = 1024, kBatchMaxGemvs = 1024, kBatchMaxItems = 65536;

size_t batch_block_bytes() {
    return round_up(sizeof(DGemm) * kBatchMaxGemms, 256) +
           round_up(sizeof(DGemv) * kBatchMaxGemvs, 256) + sizeof(Item) * kBatchMaxItems;
}

// Resident workgroups per CU of a kind's kernel.
int kind_per_cu(Kind k) {
    static int per_cu[NKIND] = {};
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    if (per_cu[k] == 0) {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, grouped_kernel_of(k), NT, 0) !=
                hipSuccess ||
            v < 1) {
            (void)hipGetLastError();
            v = 1;
        }
        per_cu[k] = v;
    }
    return per_cu[k];
}
}  // namespace

omb_status batch_create(GroupBatch** out) {
    *out = nullptr;
    auto* b = new GroupBatch();
    b->bytes = batch_block_bytes();
    if (hipMalloc(reinterpret_cast<void**>(&b->dev), b->bytes) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&b->host), b->bytes) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&b->counters), 2 * sizeof(unsigned)) != hipSuccess ||
        hipMemset(b->counters, 0, 2 * sizeof(unsigned)) != hipSuccess) {
        (void)hipGetLastError();
        batch_destroy(b);
        set_error("serve: batch buffer allocation failed");
        return OMB_ENOMEM;
    }
    *out = b;
    return OMB_OK;
}

void batch_destroy(GroupBatch* b) {
    if (!b) return;
    if (b->dev) (void)hipFree(b->dev);
    if (b->host) (void)hipHostFree(b->host);
    if (b->counters) (void)hipFree(b->counters);
    delete b;
}

bool batch_mode_supported(int mode) {
    return mode == OMB_MODE_PLAIN_F32 || mode == OMB_MODE_SPLIT_BF16 ||
           mode == OMB_MODE_SPLIT_BF16_P3;
}

omb_status batch_launch(GroupBatch* b, const omb_gemm_desc* gemms, int n_gemm,
                        const omb_gemv_desc* gemvs, int n_gemv, int mode, hipStream_t s) {
    if (!batch_mode_supported(mode)) {
        set_error("serve batch: mode " + std::to_string(mode) + " is not batched");
        return OMB_EUNSUPPORTED;
    }
    if (n_gemm < 0 || n_gemv < 0 || n_gemm > kBatchMaxGemms || n_gemv > kBatchMaxGemvs) {
        set_error("serve batch: too many instances");
        return OMB_EUNSUPPORTED;
    }
    OMB_TRY(validate(gemms, n_gemm, gemvs, n_gemv));
    DGemm* g = reinterpret_cast<DGemm*>(b->host);
    const size_t voff = round_up(sizeof(DGemm) * kBatchMaxGemms, 256);
    DGemv* v = reinterpret_cast<DGemv*>(b->host + voff);
    const size_t ioff = voff + round_up(sizeof(DGemv) * kBatchMaxGemvs, 256);
    Item* items = reinterpret_cast<Item*>(b->host + ioff);
    std::vector<Item> list;
    std::vector<DGemm> gv(n_gemm);
    std::vector<DGemv> vv(n_gemv);
    for (int i = 0; i < n_gemm; ++i) {
        const omb_gemm_desc& d = gemms[i];
        gv[i] = DGemm{d.M, d.N, d.K, d.A, d.lda, d.B, d.ldb, d.C, d.ldc, d.alpha, d.beta,
                      nullptr, nullptr};
        if (d.M == 0 || d.N == 0) continue;
        int c = choose_class(mode, d);
        if (c == C128x64) c = C64;  // same bits; keeps the lite kernel
        const int64_t tmn = ceil_div(d.M, kTileM[c]), tnn = ceil_div(d.N, kTileN[c]);
        if ((int64_t)list.size() + tmn * tnn > kBatchMaxItems) {
            set_error("serve batch: too many tiles");
            return OMB_EUNSUPPORTED;
        }
        for (int64_t a = 0; a < tmn; ++a)
            for (int64_t bb = 0; bb < tnn; ++bb) list.push_back(Item{c, i, (int)a, (int)bb});
    }
    for (int i = 0; i < n_gemv; ++i) {
        const omb_gemv_desc& d = gemvs[i];
        vv[i] = DGemv{d.M, d.N, d.A, d.lda, d.x, d.y, d.alpha, d.beta};
        const int64_t chunks = ceil_div(d.M, 64);
        if ((int64_t)list.size() + chunks > kBatchMaxItems) {
            set_error("serve batch: too many GEMV chunks");
            return OMB_EUNSUPPORTED;
        }
        for (int64_t c = 0; c < chunks; ++c) list.push_back(Item{CGEMV, i, (int)c, 0});
    }
    const int nitems = (int)list.size();
    if (nitems == 0) return OMB_OK;
    std::vector<double> cost(list.size());
    for (size_t i = 0; i < list.size(); ++i) cost[i] = item_cost(list[i], gv, vv);
    std::vector<size_t> order(list.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(),
                     [&](size_t x, size_t y) { return cost[x] > cost[y]; });
    if (n_gemm) std::memcpy(g, gv.data(), sizeof(DGemm) * n_gemm);
    if (n_gemv) std::memcpy(v, vv.data(), sizeof(DGemv) * n_gemv);
    for (size_t i = 0; i < order.size(); ++i) items[i] = list[order[i]];
    // One copy of the used block (the unused tails of the descriptor arrays
    // travel too; the block is at most a few hundred KB).
    const size_t used = ioff + sizeof(Item) * (size_t)nitems;
    OMB_HIP_TRY(hipMemcpyAsync(b->dev, b->host, used, hipMemcpyHostToDevice, s));
    const Kind kind = kind_of(mode, false);
    const int grid = std::max(1, std::min(nitems, device_cu_count() * kind_per_cu(kind)));
    const int chunk = std::max(1, std::min(4, nitems / (8 * grid)));
    PArgs a{reinterpret_cast<const Item*>(b->dev + ioff), nitems,
            reinterpret_cast<const DGemm*>(b->dev), reinterpret_cast<const DGemv*>(b->dev + voff),
            b->counters, chunk, (int)ceil_div(nitems, chunk)};
    hipLaunchKernelGGL(grouped_kernel_of(kind), dim3(grid), dim3(NT), 0, s, a);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

// The steps of batch_launch over no items: the occupancy query (cached for
// the process), a copy of the whole pinned block (copies this size run as a
// runtime kernel, whose first launch is the cost), and each kind's launch, in which one
// workgroup finds no chunk (nchunks = 0), reads no item and, as the last
// workgroup to finish, leaves both counters at zero.
omb_status batch_warm(GroupBatch* b, hipStream_t s) {
    OMB_HIP_TRY(hipMemcpyAsync(b->dev, b->host, b->bytes, hipMemcpyHostToDevice, s));
    PArgs a{reinterpret_cast<const Item*>(b->dev), 0, reinterpret_cast<const DGemm*>(b->dev),
            reinterpret_cast<const DGemv*>(b->dev), b->counters, 1, 0};
    for (int mode : {OMB_MODE_PLAIN_F32, OMB_MODE_SPLIT_BF16, OMB_MODE_SPLIT_BF16_P3}) {
        const Kind kind = kind_of(mode, false);  // the modes batch_launch takes
        (void)kind_per_cu(kind);
        hipLaunchKernelGGL(grouped_kernel_of(kind), dim3(1), dim3(NT), 0, s, a);
        OMB_HIP_TRY(hipGetLastError());
    }
    return OMB_OK;
}

}  // namespace omb
