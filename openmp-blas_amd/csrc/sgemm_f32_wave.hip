// Plain FP32 SGEMM for products whose 128x128 tiles leave CUs idle: C =
// alpha*A*B + beta*C with K divided among the wavefronts of a workgroup.
//
// Counterpart of the same code as sgemm_f32.hip (include/mtm.hpp:83-206,
// include/simd_loop.hpp:80-192), for the small and middle sizes of the
// reference's sweep (src/mtm.cpp:372-375).  A workgroup of W wavefronts owns
// one BM x BN tile of C.  Wavefront w sums the 128-k accumulation blocks w,
// w + W, ... of the whole tile, each from zero, with 4*GR x 4*GC outputs per
// lane; after every W blocks the wavefronts' block sums meet in LDS and are
// added to the tile in block order.  That is the unsplit kernel's own fold,
// outer = ((b0 + b1) + b2) ..., and where the tile classes would split K in
// coarser pieces, whose sums are shorter and err less, the fold starts anew at
// every piece and the pieces' sums (kept in LDS) are added in order.  So the
// bits are those of sgemm_f32_kernel with that split for any W and K, with no
// partial sums in memory and no second launch, and a wavefront holds one
// accumulator tile instead of two.
//
// Each wavefront stages its own 16-k slices of A and B through its own LDS
// buffers (LDS operations of a wavefront complete in order, so the k loop has
// no workgroup barrier), with the next slice's global loads in flight.  Rows and
// columns past C are clamped to valid addresses: what they give is never
// stored.  Only K's last slice (and the last slice of a tile whose 4-column
// loads could pass the end of an operand) loads element by element.
//
// Bound by FP32 issue once the chip is full; below that by the launch and one
// memory round trip per slice.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "sgemm_wave.hpp"

namespace omb {
namespace {

using namespace wave;

constexpr int kGroupM = 8;

struct WArgs {
    int64_t M, N, K;
    float alpha, beta;
    const float* A;
    int64_t lda;
    const float* B;
    int64_t ldb;
    float* C;
    int64_t ldc;
    int64_t tiles_m, tiles_n;
    int seg;  // accumulation blocks per piece of K, or 0: K is one piece
};

// GR, GC: 4-row and 4-column groups per lane (8 x 8 lanes: BM = 32*GR, BN =
// 32*GC); W wavefronts.  PIECES: K is folded in pieces of p.seg blocks; a build of
// its own, since the code for them made products of few k up to 7% slower
// (1150 x 1310 x 33: 8.2 us, 8.8 with one build for both).
template <int GR, int GC, int W, int OCC, bool PIECES, bool A_KC, bool B_NC, typename Off>
__global__ __launch_bounds__(64 * W, OCC) void sgemm_f32_wave_kernel(WArgs p) {
    static_assert(W > 1, "the wavefronts share K");
    constexpr int BM = 32 * GR, BN = 32 * GC, TR = 4 * GR;
    constexpr int S = TR * GC;            // float4 of the tile per lane
    constexpr int P = S > 4 ? 2 : 1;      // passes of the LDS sum (bounds its LDS)
    constexpr int SP = S / P, OWN = (SP + W - 1) / W;  // float4 per pass; of them, added here
    union Shared {
        WaveStage<GR, GC> stage[W];
        acc4 sum[W][SP][64];
    };
    __shared__ __attribute__((aligned(16))) Shared sh;
    __shared__ acc4 total[PIECES ? P * OWN : 1][PIECES ? 64 * W : 1];  // the pieces' sums, each thread's own

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lx = lane & 7, ly = lane >> 3;
    int64_t tm, tn;
    group_tile(xcd_remap(blockIdx.x, (unsigned)(p.tiles_m * p.tiles_n)), p.tiles_m, p.tiles_n, kGroupM, &tm, &tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;
    WaveSide<BM, A_KC, Off, const float*> sa;
    WaveSide<BN, !B_NC, Off, const float*> sb;
    sa.init(p.A, p.lda, m0, p.M, lane);
    sb.init(p.B, p.ldb, n0, p.N, lane);
    Off oa[sa.L], ob[sb.L];
#pragma unroll
    for (int i = 0; i < sa.L; ++i) oa[i] = sa.offset(i);
#pragma unroll
    for (int i = 0; i < sb.L; ++i) ob[i] = sb.offset(i);
    const int tail = max(sa.tail(), sb.tail());

    acc4 inner[TR][GC];
    WaveStage<GR, GC>& st = sh.stage[wave];
    auto compute = [&] { wave_compute<GR, GC>(st, lane, inner); };

    acc4 outer[P * OWN];
#pragma unroll
    for (int o = 0; o < P * OWN; ++o) outer[o] = acc4{0.f, 0.f, 0.f, 0.f};
    const int64_t nblk = ceil_div(p.K, BLOCK_K);
    int left = p.seg;  // blocks until the piece ends
    for (int64_t first = 0; first < nblk; first += W) {
        const int64_t blk = first + wave;
        if (blk < nblk) {
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int h = 0; h < GC; ++h) inner[i][h] = acc4{0.f, 0.f, 0.f, 0.f};
            const int64_t kb = blk * BLOCK_K, ke = std::min<int64_t>(p.K, kb + BLOCK_K);
            const int nfull = full_slices((int)(ke - kb), p.K - ke, tail);
            const int64_t klast = kb + (int64_t)std::max(nfull - 1, 0) * BK;
            float4 va[sa.L], vb[sb.L];
            auto load = [&](int64_t k) {
                k = k < klast ? k : klast;
                sa.load(va, oa, k);
                sb.load(vb, ob, k);
            };
            auto store = [&] {
                wave_lds_fence();
                sa.store(st.a, va);
                sb.store(st.b, vb);
                wave_lds_fence();
            };
            int s = 0;
            if (nfull > 1) {
                load(kb);
                store();
                for (; s < nfull; ++s) {  // slice s is staged
                    pin(inner);
                    load(kb + (int64_t)(s + 1) * BK);
                    __builtin_amdgcn_sched_barrier(0);
                    compute();
                    store();
                }
            }
            // a lone slice, and what unguarded loads leave: K % 16, the end of K
#pragma unroll 1
            for (int64_t k = kb + (int64_t)s * BK; k < ke; k += BK, ++s) {
                if (s < nfull) {
                    load(k);
                } else {
                    sa.load_guarded(va, k, std::min<int64_t>(ke, k + BK));
                    sb.load_guarded(vb, k, std::min<int64_t>(ke, k + BK));
                }
                store();
                compute();
            }
        }
        // Block sums -> LDS, added in block order by the wavefront that owns
        // each float4 of the lanes' tiles.
        const int in_round = (int)std::min<int64_t>(W, nblk - first);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            __syncthreads();  // the staging buffers, or the last pass, are read
            if (wave < in_round) {
#pragma unroll
                for (int s = 0; s < SP; ++s)
                    sh.sum[wave][s][lane] = inner[(q * SP + s) / GC][(q * SP + s) % GC];
            }
            __syncthreads();
            int until = left;
            for (int w = 0, e; w < in_round; w = e) {
                e = PIECES ? std::min(in_round, w + until) : in_round;
                for (int b = w; b < e; ++b) {
#pragma unroll
                    for (int o = 0; o < OWN; ++o) {
                        const int slot = wave * OWN + o;
                        if (slot >= SP) continue;
                        outer[q * OWN + o] += sh.sum[b][slot][lane];
                    }
                }
                if constexpr (PIECES) {
                    until -= e - w;
                    if (until > 0) continue;
                    until = p.seg;
#pragma unroll
                    for (int o = 0; o < OWN; ++o) {
                        acc4& t = total[q * OWN + o][threadIdx.x];
                        t = first + e == p.seg ? outer[q * OWN + o] : t + outer[q * OWN + o];
                        outer[q * OWN + o] = acc4{0.f, 0.f, 0.f, 0.f};
                    }
                }
            }
            if (q == P - 1) left = until;
        }
        if (first + W < nblk) __syncthreads();  // before the next round's staging
    }

    if constexpr (PIECES) {  // K has more than one
#pragma unroll
        for (int o = 0; o < P * OWN; ++o) outer[o] += total[o][threadIdx.x];
    }
    // Whole quads at any alignment, the reads of C ahead of the writes.
    const int rows = (int)std::min<int64_t>(p.M - m0, BM), cols = (int)std::min<int64_t>(p.N - n0, BN);
    float* const c0 = p.C + m0 * p.ldc + n0;
    auto place = [&](int o, int* m, int* n) {  // outer[o]'s row and first column
        const int in_pass = wave * OWN + o % OWN, slot = o / OWN * SP + in_pass;
        *m = (slot / GC >> 2) * 32 + ly * 4 + (slot / GC & 3);
        *n = slot % GC * 32 + lx * 4;
        return in_pass < SP && *m < rows && *n < cols;
    };
    float4 old[P * OWN];
    if (p.beta != 0.f) {
#pragma unroll
        for (int o = 0; o < P * OWN; ++o) {
            int m, n;
            if (place(o, &m, &n) && n + 3 < cols) old[o] = ld4u(c0 + m * p.ldc + n);
        }
    }
#pragma unroll
    for (int o = 0; o < P * OWN; ++o) {
        int m, n;
        if (!place(o, &m, &n)) continue;
        float* c = c0 + m * p.ldc + n;
        f32x4_u v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = p.alpha * outer[o][acc_slot(e)];
        if (n + 3 < cols) {
            if (p.beta != 0.f)
                v = f32x4_u{v[0] + p.beta * old[o].x, v[1] + p.beta * old[o].y,
                            v[2] + p.beta * old[o].z, v[3] + p.beta * old[o].w};
            *reinterpret_cast<f32x4_u*>(c) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < cols) c[e] = p.beta != 0.f ? v[e] + p.beta * c[e] : v[e];
        }
    }
}

// The classes: tile, wavefronts, and the measured model of a launch's time (us):
//   fixed + the rounds of W blocks one after another at `block` us each, or
//   fixed + the tiles' flop at `rate` TFLOP/s, an idle wavefront of the last
//   round costing `idle` of a busy one and the last wave of workgroups (per_cu
//   resident per CU) its square root of unevenness, whichever is longer.
// Fitted to 1120 products with M, N and K from 32 to 6144 (geometrically drawn, up to 4e10
// flop): with the choice of sgemm_f32_choose they took 1/1.22 of the tile classes'
// time, against 1/1.23 if the fastest were always chosen.

struct WaveClass {
    int gr, gc, w, per_cu;
    double fixed, rate, block, idle;
};
constexpr WaveClass kWaveClasses[4] = {
    {2, 2, 8, 1, 5.0, 72.0, 15.0, 0.35},
    {1, 1, 8, 2, 3.1, 49.0, 7.8, 0.46},
    {1, 1, 4, 5, 3.0, 64.0, 8.4, 0.30},
    {1, 1, 2, 10, 4.7, 78.0, 9.9, 0.31},
};

template <int GR, int GC, int W, int OCC>
void launch_class(const WArgs& p, bool a_kc, bool b_nc, hipStream_t s) {
    const bool near = offsets_fit32(a_kc, p.lda, std::min<int64_t>(p.M, 32 * GR)) &&
                      offsets_fit32(!b_nc, p.ldb, std::min<int64_t>(p.N, 32 * GC));
    auto pick = [&](auto off, auto pieces) {
        using Off = decltype(off);
        constexpr bool P = decltype(pieces)::value;
        return a_kc ? (b_nc ? sgemm_f32_wave_kernel<GR, GC, W, OCC, P, true, true, Off>
                            : sgemm_f32_wave_kernel<GR, GC, W, OCC, P, true, false, Off>)
                    : (b_nc ? sgemm_f32_wave_kernel<GR, GC, W, OCC, P, false, true, Off>
                            : sgemm_f32_wave_kernel<GR, GC, W, OCC, P, false, false, Off>);
    };
    const std::true_type yes;
    const std::false_type no;
    const auto kernel = p.seg ? (near ? pick(0u, yes) : pick((int64_t)0, yes))
                              : (near ? pick(0u, no) : pick((int64_t)0, no));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(64 * W), 0, s, p);
}

}  // namespace

int sgemm_f32_wave_class(int64_t M, int64_t N, int64_t K, double* time) {
    int best = -1;
    for (int c = 0; c < 4; ++c) {
        const WaveClass& k = kWaveClasses[c];
        const double bm = 32 * k.gr, bn = 32 * k.gc;
        const int64_t tiles = ceil_div(M, (int64_t)bm) * ceil_div(N, (int64_t)bn);
        const int64_t blocks = ceil_div(K, BLOCK_K), rounds = ceil_div(blocks, k.w);
        const double busy = (double)K / BLOCK_K + k.idle * (double)(rounds * k.w - blocks);
        const double r = (double)tiles / ((double)k.per_cu * device_cu_count());
        const double full = 2.0 * bm * bn * BLOCK_K * (double)tiles * busy / (k.rate * 1e6) *
                            (r >= 1.0 && r < 4.0 ? std::sqrt(std::ceil(r) / r) : 1.0);
        const double chain = (double)rounds * k.block * std::min(1.0, (double)K / BLOCK_K);
        const double t = (k.fixed + std::max(chain, full)) * 1e-6;
        if (tiles * 64 * k.w < kLaunchItems && t < *time) {
            best = c;
            *time = t;
        }
    }
    return best;
}

omb_status launch_sgemm_f32_wave(int cls, int64_t M, int64_t N, int64_t K, float alpha,
                                 const float* A, int64_t lda, bool a_kc, const float* B,
                                 int64_t ldb, bool b_nc, float beta, float* C, int64_t ldc,
                                 int64_t kchunk, hipStream_t s) {
    const WaveClass& k = kWaveClasses[cls];
    const WArgs p{M, N, K, alpha, beta, A, lda, B, ldb, C, ldc,
                  ceil_div(M, 32 * k.gr), ceil_div(N, 32 * k.gc),
                  kchunk < K && kchunk > BLOCK_K ? (int)(kchunk / BLOCK_K) : 0};
    if (cls == 0) launch_class<2, 2, 8, 1>(p, a_kc, b_nc, s);
    else if (cls == 1) launch_class<1, 1, 8, 2>(p, a_kc, b_nc, s);
    else if (cls == 2) launch_class<1, 1, 4, 5>(p, a_kc, b_nc, s);
    else launch_class<1, 1, 2, 5>(p, a_kc, b_nc, s);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

}  // namespace omb
