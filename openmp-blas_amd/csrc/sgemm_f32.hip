// Plain FP32 SGEMM for gfx950: C = alpha*A*B + beta*C on the vector ALUs.
//
// Counterpart of amt::mtm_helper / impl::mtm_kernel / simd_loop<MTM>
// (include/mtm.hpp:83-206, include/simd_loop.hpp:80-192): the reference packs
// MR x KC and KC x NR panels into cache-sized buffers and runs a 16x6 register
// micro-kernel.  Here a 256-thread workgroup owns a BM x BN tile of C (three
// classes: 128x128, 128x64, 64x64 -- a3's cache-level block choice becomes a
// choice of tile class and K split per shape), stages BM x 16 and 16 x BN
// slices of A and B through LDS (double buffered; the staging plays the role
// of `pack`, including the layout change for either operand order), and
// every thread keeps a (BM/16) x (BN/16) register micro-tile.  Global loads
// run two slices ahead in registers and LDS fragments one k ahead.
//
// What bounds it: the issue of v_fmac_f32, 128 per CU and clock.  Two things
// keep the k loop near it (4096^3 in us by layout of A and B, row.row, col.row,
// row.col, col.col: 1538 1539 1453 1547 without them, 1429 1423 1447 1436 with):
//  - every full slice of every tile is read with unguarded 128-bit loads at any
//    alignment, addressed by a uniform base and 32-bit byte offsets (see Side);
//    ragged tiles took guarded loads before, 1.05-1.36x the time;
//  - an accumulator never lies in the register bank of the B value it is
//    multiplied with (registers r and r + 4n share a bank, and a v_fmac with two
//    operands in one bank takes a cycle more): the four accumulators of a B quad
//    are one 4-register tuple, rotated by one against the quad (acc_slot).
//
// Accumulation order: each thread sums 128 consecutive k (8 LDS slices) into
// an inner register tile, then adds it to an outer tile -- the same for every
// tile class, so the class never changes an output's bits.  This two-level sum
// keeps the rounding error of long K at or below the reference's (which sums
// KC consecutive k and then does C += block, simd_loop.hpp:120-128,160-190).
//
// Row-major C only: a column-major C is handled by the caller through
// C^T = B^T A^T (swap operands and their strides).
#include "slice_bounds.hpp"

namespace omb {
namespace {

constexpr int BK = kSliceK;
constexpr int NT = 256;         // threads per workgroup (a 16 x 16 thread grid)
constexpr int INNER_K = 128;    // k steps per inner accumulation block
constexpr int PAD = 4;          // LDS row padding (floats), keeps float4 alignment
constexpr int kGroupM = 8;      // tile rows per L2 group
constexpr int64_t kSplitMinK = 256;    // least k per coarse split (K > kSplitExactK)
constexpr int64_t kSplitExactK = 512;  // up to this K, splits are only single accumulation blocks
constexpr int64_t kSplitMost = 16;     // most coarse splits considered
constexpr double kSplitMaxBytes = 128.0 * (1 << 20);  // most partial-sum bytes
// FP32 flop/s of one 128x128 workgroup, measured: with two per CU (86
// TFLOP/s over 512 at 8192^3) and alone on its CU (50 TFLOP/s over 256 at
// 2048^3: one wave per SIMD loses the dual issue of two).
constexpr double kTileRateF32 = 0.17e12;
constexpr double kTileRateF32Alone = 0.2e12;
// The same for the 128x64 class (three per CU) and the 64x64 class (four
// per CU), scaled from one measurement of all three classes (8192 x 8192 x
// 2048 for the full rate, 16 x 16 tiles with K = 4096 alone): per workgroup
// 0.154 / 0.103 / 0.072 TFLOP/s full and 0.196 / 0.155 / 0.126 alone.
constexpr double kTileRateF32_128x64 = 0.114e12;
constexpr double kTileRateF32_128x64Alone = 0.158e12;
constexpr double kTileRateF32_64x64 = 0.079e12;
constexpr double kTileRateF32_64x64Alone = 0.129e12;
// A product's time by the tile classes, for the comparison with the classes of
// sgemm_f32_wave.hip: launch (with a split's second one) and scale of the model.
constexpr double kTileLaunch = 6.4e-6, kTileScale = 0.78;
constexpr double kSplitHbm = 4.0e12;      // bytes/s for the partials' traffic
constexpr double kSplitLaunch = 4.0e-6;   // the reduction kernel's launch and tail
constexpr double kSplitReduceStep = 1.0e-6;  // one round trip per 8 partials of an element

struct Args {
    int64_t M, N, K;
    float alpha, beta;
    const float* A;
    int64_t lda;
    const float* B;
    int64_t ldb;
    float* C;
    int64_t ldc;
    int64_t tiles_m, tiles_n;
    int64_t kchunk;  // k per split (blockIdx.y), a multiple of INNER_K
    float* part;     // split partial sums [split][M][N], or null (one split)
};

// One operand's side of a workgroup's tile: E lines (rows of A or columns of
// B) from line e0 of the operand; KC: k is the unit stride, else the line is.
// Its 16-k slices are read with 128-bit loads along the unit stride at any
// alignment, whose lines are clamped into the operand instead of guarded: what
// the repeated lines give is never stored, so every full slice of every tile,
// ragged or not, takes the same unguarded loads.  A thread's loads are byte
// offsets from the slice's first element, of 32 bits unless the leading
// dimension is too long for that (offsets_fit32).
template <int E, bool KC, typename Off>
struct Side {
    static constexpr int L = E / 64;  // float4 per thread and slice
    const float* p;                   // line e0, this split's first k
    int64_t ld;
    int n;                            // lines from e0 inside the operand, at most E
    Off off[L];                       // this thread's loads of a slice, in bytes

    __device__ __forceinline__ void init(const float* X, int64_t ld_, int64_t e0, int64_t lines,
                                         int64_t kbeg, int tid) {
        ld = ld_;
        p = X + (KC ? e0 * ld + kbeg : e0 + kbeg * ld);
        n = (int)std::min<int64_t>(lines - e0, E);
#pragma unroll
        for (int i = 0; i < L; ++i) off[i] = (Off)(4 * slice_load<E, KC>(tid + i * NT, n, ld));
    }
    __device__ __forceinline__ int tail() const { return slice_tail<KC>(n, ld); }
    __device__ __forceinline__ void load(float4 (&v)[L], int64_t k0) const {
        const char* q = reinterpret_cast<const char*>(p + (KC ? k0 : k0 * ld));
#pragma unroll
        for (int i = 0; i < L; ++i) v[i] = ld4u(reinterpret_cast<const float*>(q + off[i]));
    }
    // Registers -> LDS, laid out [k][line].
    __device__ __forceinline__ void store(float (*s)[E + PAD], const float4 (&v)[L], int tid) const {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int e = tid + i * NT;
            if (KC) {
                const int line = e >> 2, kq = (e & 3) * 4;
                s[kq + 0][line] = v[i].x;
                s[kq + 1][line] = v[i].y;
                s[kq + 2][line] = v[i].z;
                s[kq + 3][line] = v[i].w;
            } else {
                *reinterpret_cast<float4*>(&s[e / (E / 4)][e % (E / 4) * 4]) = v[i];
            }
        }
    }
    // The slice at k0 with kn valid k, element by element: zeros past them.
    __device__ __forceinline__ void stage_tail(float (*s)[E + PAD], int64_t k0, int kn, int tid) const {
#pragma unroll 4
        for (int e = tid; e < E * BK; e += NT) {
            const int line = KC ? e / BK : e % E, k = KC ? e % BK : e / E;
            const int a = min(line, n - 1);
            const int64_t b = k0 + min(k, kn - 1);
            const float x = p[KC ? a * ld + b : b * ld + a];
            s[k][line] = k < kn ? x : 0.f;
        }
    }
};

// Workgroups per CU each class is built for: the 128x128 class holds 2 x 64
// accumulators per thread (2 workgroups per CU), 128x64 2 x 32 (3), 64x64
// 2 x 16 (4).
constexpr int occ_of(int tile_elems) {
    return tile_elems >= 128 * 128 ? 2 : (tile_elems >= 128 * 64 ? 3 : 4);
}

// Thread (ty, tx) of the 16 x 16 grid owns rows {g*64 + ty*4 + i} (g < GR =
// BM/64, i < 4) and columns {h*64 + tx*4 + j} (h < GC = BN/64, j < 4).
template <int BM, int BN, bool A_KC, bool B_NC, typename Off>
__global__ __launch_bounds__(NT, occ_of(BM * BN)) void sgemm_f32_kernel(Args q) {
    constexpr int GR = BM / 64, GC = BN / 64, TR = 4 * GR;
    __shared__ float As[2][BK][BM + PAD];
    __shared__ float Bs[2][BK][BN + PAD];

    // Split blockIdx.y takes k in [y * kchunk, min(K, (y + 1) * kchunk)): the
    // operands are offset to that range and K becomes its length.  kchunk is
    // a multiple of INNER_K, so the 128-k accumulation blocks are the same
    // as without the split.
    Args p = q;
    const int64_t kbeg = q.part ? (int64_t)blockIdx.y * q.kchunk : 0;
    if (q.part) p.K = q.K - kbeg < q.kchunk ? q.K - kbeg : q.kchunk;

    const int tid = threadIdx.x;
    const int64_t ntiles = p.tiles_m * p.tiles_n;
    const unsigned t = xcd_remap(blockIdx.x, (unsigned)ntiles);
    int64_t tm, tn;
    group_tile(t, p.tiles_m, p.tiles_n, kGroupM, &tm, &tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;

    const int tx = tid & 15, ty = tid >> 4;
    acc4 inner[TR][GC], outer[TR][GC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int h = 0; h < GC; ++h) inner[i][h] = outer[i][h] = acc4{0.f, 0.f, 0.f, 0.f};

    const int64_t nk = ceil_div(p.K, BK);
    constexpr int kFold = INNER_K / BK;
    // Slices kt and kt+1 live in LDS buffers 0 and 1; global loads run two
    // slices ahead in two register sets.
    auto compute = [&](int cur, int64_t kt) {
        float4 fa[2][GR], fb[2][GC];
        auto fragment = [&](int k, int set) {
#pragma unroll
            for (int g = 0; g < GR; ++g)
                fa[set][g] = *reinterpret_cast<const float4*>(&As[cur][k][g * 64 + ty * 4]);
#pragma unroll
            for (int h = 0; h < GC; ++h)
                fb[set][h] = *reinterpret_cast<const float4*>(&Bs[cur][k][h * 64 + tx * 4]);
        };
        fragment(0, 0);
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            if (k + 1 < BK) fragment(k + 1, (k + 1) & 1);
            float a[TR];
#pragma unroll
            for (int g = 0; g < GR; ++g) {
                const float4 v = fa[k & 1][g];
                a[4 * g] = v.x; a[4 * g + 1] = v.y; a[4 * g + 2] = v.z; a[4 * g + 3] = v.w;
            }
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int h = 0; h < GC; ++h) {
                    const float4 v = fb[k & 1][h];
                    acc4& s = inner[i][h];
                    s[acc_slot(0)] = fmaf(a[i], v.x, s[acc_slot(0)]);
                    s[acc_slot(1)] = fmaf(a[i], v.y, s[acc_slot(1)]);
                    s[acc_slot(2)] = fmaf(a[i], v.z, s[acc_slot(2)]);
                    s[acc_slot(3)] = fmaf(a[i], v.w, s[acc_slot(3)]);
                }
        }
        if ((kt + 1) % kFold == 0 || kt + 1 == nk) {
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int h = 0; h < GC; ++h) {
                    outer[i][h] += inner[i][h];
                    inner[i][h] = acc4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    // The slices whose loads cannot pass an operand's end, then the rest (K's
    // last partial slice, or the last one of a tile with a partial quad of
    // lines) element by element.
    Side<BM, A_KC, Off> sa;
    Side<BN, !B_NC, Off> sb;
    sa.init(p.A, p.lda, m0, p.M, kbeg, tid);
    sb.init(p.B, p.ldb, n0, p.N, kbeg, tid);
    // (in 32 bits: in 64 the accumulators of one slice in two moved to B's register
    // banks, and 8192^3 took 0.4% longer)
    const int after = (int)std::min<int64_t>(q.K - kbeg - p.K, BK);
    const int64_t nfull = full_slices(p.K, after, max(sa.tail(), sb.tail()));
    int64_t kt = 0;
    if (nfull > 0) {
        // Slices kt and kt+1 in LDS buffers 0 and 1, loads two slices ahead in
        // two register sets with the slice index clamped to the last one, in
        // whole slice pairs: one path through the loop keeps the compiler's
        // wait counts exact (a store waits only for its own loads).
        float4 ra0[sa.L], rb0[sb.L], ra1[sa.L], rb1[sb.L];
        const int64_t klast = nfull - 1;
        auto kc = [&](int64_t k) { return (k < klast ? k : klast) * BK; };
        sa.load(ra0, 0);
        sb.load(rb0, 0);
        sa.store(As[0], ra0, tid);
        sb.store(Bs[0], rb0, tid);
        sa.load(ra1, kc(1));
        sb.load(rb1, kc(1));
        __syncthreads();
        for (; kt + 1 < nfull; kt += 2) {
            // Keeps each tuple in four consecutive registers through the loop.
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int h = 0; h < GC; ++h) asm volatile("" : "+v"(inner[i][h]));
            sa.load(ra0, kc(kt + 2));
            sb.load(rb0, kc(kt + 2));
            __builtin_amdgcn_sched_barrier(0);
            compute(0, kt);
            sa.store(As[1], ra1, tid);
            sb.store(Bs[1], rb1, tid);
            __syncthreads();
            sa.load(ra1, kc(kt + 3));
            sb.load(rb1, kc(kt + 3));
            __builtin_amdgcn_sched_barrier(0);
            compute(1, kt + 1);
            sa.store(As[0], ra0, tid);
            sb.store(Bs[0], rb0, tid);
            __syncthreads();
        }
    }
    // Buffer 0 holds an odd last full slice, if there is one.
    for (; kt < nk; ++kt) {
        if (kt >= nfull) {
            const int kn = (int)std::min<int64_t>(BK, p.K - kt * BK);
            sa.stage_tail(As[0], kt * BK, kn, tid);
            sb.stage_tail(Bs[0], kt * BK, kn, tid);
            __syncthreads();
        }
        compute(0, kt);
        __syncthreads();
    }

    // Epilogue: rows {g*64 + ty*4 + i}, columns {h*64 + tx*4 + j}, whole quads
    // with 128-bit accesses at any alignment, the reads of C in one batch ahead
    // of the writes.  This bounds products of few k: 5949 x 3823 x 57 with beta
    // = 1 took 119 us with element accesses on its unaligned rows, 91 with
    // quads, 78 with the reads ahead; 8192 x 8192 x 64: 228, 225, 171.
    const int rows = (int)std::min<int64_t>(p.M - m0, BM), cols = (int)std::min<int64_t>(p.N - n0, BN);
    if (p.part) {  // raw partial sums of this split, row-major M x N
        float* const c0 = p.part + ((int64_t)blockIdx.y * p.M + m0) * p.N + n0;
#pragma unroll
        for (int i = 0; i < TR; ++i)
#pragma unroll
            for (int h = 0; h < GC; ++h) {
                const int m = (i / 4) * 64 + ty * 4 + (i % 4), n = h * 64 + tx * 4;
                if (m >= rows) continue;
                float* c = c0 + m * p.N + n;
                const acc4 v = outer[i][h];
                if (n + 3 < cols)
                    *reinterpret_cast<f32x4_u*>(c) = f32x4_u{v[acc_slot(0)], v[acc_slot(1)],
                                                             v[acc_slot(2)], v[acc_slot(3)]};
                else
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (n + j < cols) c[j] = v[acc_slot(j)];
            }
        return;
    }
    const float alpha = p.alpha, beta = p.beta;
    const int64_t ldo = p.ldc;
    float* const c0 = p.C + m0 * ldo + n0;
    float4 old[TR][GC];
    if (beta != 0.f) {
#pragma unroll
        for (int i = 0; i < TR; ++i)
#pragma unroll
            for (int h = 0; h < GC; ++h) {
                const int m = (i / 4) * 64 + ty * 4 + (i % 4), n = h * 64 + tx * 4;
                if (m < rows && n + 3 < cols) old[i][h] = ld4u(c0 + m * ldo + n);
            }
    }
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int h = 0; h < GC; ++h) {
            const int m = (i / 4) * 64 + ty * 4 + (i % 4), n = h * 64 + tx * 4;
            if (m >= rows) continue;
            float* c = c0 + m * ldo + n;
            f32x4_u v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = alpha * outer[i][h][acc_slot(j)];
            if (n + 3 < cols) {
                if (beta != 0.f)
                    v = f32x4_u{v[0] + beta * old[i][h].x, v[1] + beta * old[i][h].y,
                                v[2] + beta * old[i][h].z, v[3] + beta * old[i][h].w};
                *reinterpret_cast<f32x4_u*>(c) = v;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < cols) c[j] = beta != 0.f ? v[j] + beta * c[j] : v[j];
            }
        }
}

// C = alpha * (sum of the splits' partials, in split order) + beta * C.
// Rows over blockIdx.y, columns over threads: VEC takes four adjacent
// columns per thread with 128-bit loads and stores (N, ldc multiples of 4,
// C 16-byte aligned), else one column.  Eight partials are in flight per
// step (a long split list is otherwise one memory round trip per partial);
// every element's adds stay in split order, so VEC changes no bits.
template <bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(int64_t M, int64_t N, int64_t splits,
                                                            float alpha, float beta,
                                                            const float* __restrict__ part,
                                                            float* C, int64_t ldc) {
    constexpr int W = VEC ? 4 : 1;
    typedef float vf __attribute__((ext_vector_type(W)));
    const int64_t total = M * N, cols = N / W;
    for (int64_t m = blockIdx.y; m < M; m += gridDim.y) {
        for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < cols;
             q += (int64_t)gridDim.x * blockDim.x) {
            const int64_t i = m * N + q * W;
            vf s = *reinterpret_cast<const vf*>(part + i);
            int64_t t = 1;
            for (; t + 8 <= splits; t += 8) {
                vf v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const vf*>(part + (t + u) * total + i);
#pragma unroll
                for (int u = 0; u < 8; ++u) s += v[u];
            }
            for (; t < splits; ++t) s += *reinterpret_cast<const vf*>(part + t * total + i);
            vf* c = reinterpret_cast<vf*>(C + m * ldc + q * W);
            const vf v = alpha * s;
            *c = beta != 0.f ? v + beta * *c : v;
        }
    }
}

template <int BM, int BN, typename Off>
void launch_class(const Args& a, bool a_kc, bool b_nc, int64_t splits, hipStream_t s) {
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)splits);
    const auto kernel = a_kc ? (b_nc ? sgemm_f32_kernel<BM, BN, true, true, Off>
                                     : sgemm_f32_kernel<BM, BN, true, false, Off>)
                             : (b_nc ? sgemm_f32_kernel<BM, BN, false, true, Off>
                                     : sgemm_f32_kernel<BM, BN, false, false, Off>);
    hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, s, a);
}

template <int BM, int BN>
void launch_class(const Args& a, bool a_kc, bool b_nc, int64_t splits, hipStream_t s) {
    if (offsets_fit32(a_kc, a.lda, std::min<int64_t>(a.M, BM)) &&
        offsets_fit32(!b_nc, a.ldb, std::min<int64_t>(a.N, BN)))
        launch_class<BM, BN, unsigned>(a, a_kc, b_nc, splits, s);
    else
        launch_class<BM, BN, int64_t>(a, a_kc, b_nc, splits, s);
}

// The plain tile classes: tile shape, workgroups per CU, and the FP32 flop/s
// of one workgroup with the CU full of its class and alone on its CU.
constexpr int kTileClasses = 3;
struct F32Class {
    int bm, bn, occ;
    double rate_full, rate_alone;
};
constexpr F32Class kF32Classes[kTileClasses] = {
    {128, 128, 2, kTileRateF32, kTileRateF32Alone},
    {128, 64, 3, kTileRateF32_128x64, kTileRateF32_128x64Alone},
    {64, 64, 4, kTileRateF32_64x64, kTileRateF32_64x64Alone},
};

__global__ void scale_kernel(int64_t M, int64_t N, float beta, float* C, int64_t ldc) {
    int64_t total = M * N;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        int64_t m = i / N, n = i % N;
        float* c = C + m * ldc + n;
        *c = beta != 0.f ? beta * *c : 0.f;
    }
}

}  // namespace

int64_t gemm_k_splits_tiles(int64_t M, int64_t N, int64_t K, int64_t align, int bm, int bn,
                            int occ, double rate_full, double rate_alone, int64_t* kchunk,
                            double* time) {
    *kchunk = K;
    const int64_t tiles = ceil_div(M, bm) * ceil_div(N, bn);
    const int64_t cus = device_cu_count();
    // Rounds of workgroups (`occ` resident per CU) times the k each covers,
    // at the rate of a workgroup sharing its CU or, when there are no more
    // workgroups than CUs, alone on it; plus the partials' write and read,
    // the reduction launch and its round trips.
    auto cost = [&](int64_t splits, int64_t kc) {
        const int64_t w = tiles * splits;
        const double work = 2.0 * bm * bn * (double)kc;
        double t = w <= cus ? work / rate_alone : (double)ceil_div(w, occ * cus) * work / rate_full;
        if (splits > 1)
            t += (double)(splits + 1) * (double)(M * N) * 4.0 / kSplitHbm + kSplitLaunch +
                 (double)ceil_div(splits - 1, 8) * kSplitReduceStep;
        return t;
    };
    if (tiles <= 0 || K <= align) {
        if (time) *time = tiles > 0 ? cost(1, K) : 0.0;
        return 1;
    }
    const double part_bytes = (double)(M * N) * 4.0;
    // Exact choices first: no split, or one accumulation block per split.
    // The in-order sum of single blocks is the unsplit kernel's own fold
    // (outer = ((b0 + b1) + b2) ...), so either gives the unsplit bits, on
    // any device.  The split is taken when the model finds it 5% faster.
    int64_t best = 1;
    double best_t = cost(1, K);
    const int64_t nblk = ceil_div(K, align);
    if ((double)nblk * part_bytes <= kSplitMaxBytes) {
        const double t = cost(nblk, align);
        if (t < 0.95 * best_t) {
            best = nblk;
            best_t = t;
            *kchunk = align;
        }
    }
    if (K <= kSplitExactK) {
        if (time) *time = best_t;
        return best;
    }
    // Coarser splits (at least 256 k each) round differently: one is taken
    // only when it is more than 10% faster than the exact choice.
    const double exact_t = best_t;
    const int64_t most = std::min<int64_t>(kSplitMost, K / kSplitMinK);
    for (int64_t sp = 2; sp <= most; ++sp) {
        const int64_t kc = round_up(ceil_div(K, sp), align);
        const int64_t n = ceil_div(K, kc);
        if (kc == align) continue;  // the exact choice above
        if ((double)n * part_bytes > kSplitMaxBytes) break;  // partials too large
        const double t = cost(n, kc);
        if (n > 1 && t < 0.9 * exact_t && t < best_t) {
            best = n;
            best_t = t;
            *kchunk = kc;
        }
    }
    if (best == 1) *kchunk = K;
    if (time) *time = best_t;
    return best;
}

int64_t gemm_k_splits(int64_t M, int64_t N, int64_t K, int64_t align, double rate_full,
                      double rate_alone, int64_t* kchunk) {
    return gemm_k_splits_tiles(M, N, K, align, 128, 128, 2, rate_full, rate_alone, kchunk,
                               nullptr);
}

// Tile class and K split of a plain GEMM: the class whose modelled time is
// least, a smaller class only when the model finds it 15% faster than the
// larger one before it (with a 5% margin the model's optimism for partly
// filled rounds of small tiles cost 3-8% at some sizes from 1216 to 2432).
// Any class and any exact split give the same bits.  *time: what the model gives.
int choose_tiles(int64_t M, int64_t N, int64_t K, int64_t* splits, int64_t* kchunk,
                 double* time) {
    int best = 0;
    double best_t = 0.0;
    for (int c = 0; c < kTileClasses; ++c) {
        const F32Class& k = kF32Classes[c];
        int64_t kc = K;
        double t = 0.0;
        const int64_t sp = gemm_k_splits_tiles(M, N, K, INNER_K, k.bm, k.bn, k.occ, k.rate_full,
                                               k.rate_alone, &kc, &t);
        if (c == 0 || t < 0.85 * best_t) {
            best = c;
            best_t = t;
            *splits = sp;
            *kchunk = kc;
        }
    }
    *time = best_t;
    return best;
}

// What a product takes: a tile class with its K split, or one of the classes
// that divide K among a workgroup's wavefronts (numbered after the tiles') and
// fold its sums as that split does, whichever its model finds faster.  The tiles' model leaves out the launch and
// was fitted before their k loop gained: in this comparison their time is
// kTileLaunch + kTileScale of it, fitted with the other classes'.
int sgemm_f32_choose(int64_t M, int64_t N, int64_t K, int64_t* splits, int64_t* kchunk) {
    double t = 0.0;
    const int cls = choose_tiles(M, N, K, splits, kchunk, &t);
    t = kTileLaunch + kTileScale * t;
    const int wave = sgemm_f32_wave_class(M, N, K, &t);
    return wave < 0 ? cls : kTileClasses + wave;
}

int64_t sgemm_f32_splits(int64_t M, int64_t N, int64_t K, int64_t* kchunk) {
    int64_t splits = 1;
    double t = 0.0;
    choose_tiles(M, N, K, &splits, kchunk, &t);
    return splits;
}

omb_status launch_splitk_reduce(int64_t M, int64_t N, int64_t splits, float alpha, float beta,
                                const float* part, float* C, int64_t ldc, hipStream_t s) {
    if (M <= 0 || N <= 0) return OMB_OK;
    const bool vec = N % 4 == 0 && ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(part) & 15) == 0;
    const int64_t cols = vec ? N / 4 : N;
    const int64_t bx = std::min<int64_t>(ceil_div(cols, 256), 4 * device_cu_count());
    const int64_t by = std::min<int64_t>(
        std::min<int64_t>(M, 65535), std::max<int64_t>(1, 4 * device_cu_count() / bx));
    const dim3 grid((unsigned)bx, (unsigned)by);
    if (vec)
        hipLaunchKernelGGL(splitk_reduce_kernel<true>, grid, dim3(256), 0, s, M, N, splits, alpha,
                           beta, part, C, ldc);
    else
        hipLaunchKernelGGL(splitk_reduce_kernel<false>, grid, dim3(256), 0, s, M, N, splits,
                           alpha, beta, part, C, ldc);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

omb_status launch_sgemm_f32(int64_t M, int64_t N, int64_t K, float alpha,
                            const float* A, int64_t lda, bool a_kc,
                            const float* B, int64_t ldb, bool b_nc,
                            float beta, float* C, int64_t ldc, hipStream_t s, float* part) {
    // Tile class per shape; split K over blockIdx.y when the tiles alone
    // leave CUs idle (the splits' partials are then added in split order).
    int64_t splits = 1, kchunk = K;
    const int cls = sgemm_f32_choose(M, N, K, &splits, &kchunk);
    if (cls >= kTileClasses)
        return launch_sgemm_f32_wave(cls - kTileClasses, M, N, K, alpha, A, lda, a_kc, B, ldb, b_nc,
                                     beta, C, ldc, kchunk, s);
    const F32Class& fc = kF32Classes[cls];
    Args a{M, N, K, alpha, beta, A, lda, B, ldb, C, ldc, ceil_div(M, fc.bm), ceil_div(N, fc.bn),
           kchunk, nullptr};
    const int64_t tiles = a.tiles_m * a.tiles_n;
    if (tiles > 0x7fffffffLL) {
        set_error("sgemm: too many tiles for one launch");
        return OMB_EUNSUPPORTED;
    }
    if (splits > 1) {
        if (!part) {
            Workspace* ws = nullptr;
            OMB_TRY(get_workspace(s, (size_t)(splits * M * N) * sizeof(float), &ws));
            part = reinterpret_cast<float*>(ws->buf);
        }
        a.part = part;
    }
    if (cls == 0) launch_class<128, 128>(a, a_kc, b_nc, splits, s);
    else if (cls == 1) launch_class<128, 64>(a, a_kc, b_nc, splits, s);
    else launch_class<64, 64>(a, a_kc, b_nc, splits, s);
    OMB_HIP_TRY(hipGetLastError());
    if (splits > 1) return launch_splitk_reduce(M, N, splits, alpha, beta, a.part, C, ldc, s);
    return OMB_OK;
}

omb_status launch_scale(int64_t M, int64_t N, float beta, float* C, int64_t ldc, hipStream_t s) {
    if (M <= 0 || N <= 0 || beta == 1.f) return OMB_OK;
    int64_t total = M * N;
    unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(total, 256), 4096);
    hipLaunchKernelGGL(scale_kernel, dim3(blocks), dim3(256), 0, s, M, N, beta, C, ldc);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

}  // namespace omb
