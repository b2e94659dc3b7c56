// SGEMV for gfx950: y = alpha*A*x + beta*y, both storage orders of A.
//
// Row-major A (counterpart of mtv_helper last_order + simd_loop<INNER>,
// include/mtv.hpp:72-98, include/simd_loop.hpp:21-35): one wavefront owns
// ROWS consecutive rows; lanes stream 128-bit loads of each row, share every
// x float4 across the ROWS rows, and finish with a butterfly lane sum.
//
// Column-major A (counterpart of mtv_helper first_order + simd_loop<MTV,16>,
// include/mtv.hpp:15-70, include/simd_loop.hpp:52-78): every thread owns 4
// consecutive rows (one 128-bit load per column).  Tall matrices of whole
// 64-row blocks and 256-column rounds run in one pass of 64-row workgroups;
// otherwise the columns are split into chunks across workgroups, each chunk
// writes a partial y, and a row block's last workgroup to arrive adds its
// partials in a fixed order.
// The result depends only on (M, N) and the device's CU count, never on
// scheduling.
#include <algorithm>

#include "gemv_row.hpp"

namespace omb {
namespace {

constexpr int NT = 256;

// Rows per wavefront, 128-bit loads in flight per row and the form of the loop
// (gemv_row.hpp); the launcher chooses them.  A row's order of accumulation is
// the same for every choice.
template <int ROWS, int UNROLL, bool STREAM, bool OFF32, bool BATCH>
__global__ __launch_bounds__(NT) void sgemv_row_kernel(int64_t M, int64_t N, float alpha,
                                                       const float* __restrict__ A, int64_t lda,
                                                       const float* __restrict__ x, float beta,
                                                       float* __restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (NT / 64);
    // Grid stride over groups of ROWS rows (a grid that covers every group
    // once measured 4% slower at 16384^2 than this loop over the same grid).
    // The wavefront index is uniform: keep it (and the row pointers) scalar.
    for (int64_t w = (int64_t)blockIdx.x * (NT / 64) +
                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
         w * ROWS < M; w += waves) {
        const int64_t r0 = w * ROWS;
        const int nr = (int)std::min<int64_t>(ROWS, M - r0);
        gemv_rows_wave<ROWS, UNROLL, STREAM, OFF32, BATCH>(r0, nr, N, alpha, A, lda, x, beta, y, lane);
    }
}

// v(0) + .. + v(N - 1), added in pairs: a short product's error is that of its last
// adds, and one after the other they made it up to 1.25 times that of a sum by chunks
// alone (272 x 488: 1.12e-7 of the norm against 8.96e-8).
template <int N, typename V>
__device__ __forceinline__ float pair_sum(V v) {
    if constexpr (N == 1) return v(0);
    else return pair_sum<N / 2>(v) + pair_sum<N - N / 2>([&](int i) { return v(N / 2 + i); });
}

// Sums over a row block's chunks: a thread per row and group of consecutive chunks
// (NT / RB groups), 16 loads in flight, added in pairs as the groups are.  Thread
// t < RB returns row r0 + t's sum.
template <int RB, typename Load>
__device__ __forceinline__ float col_chunk_sum(int64_t r0, int64_t M, const float* partial,
                                               int64_t mpad, int nchunks, Load load) {
    constexpr int G = NT / RB, U = 16;
    const int per = (nchunks + G - 1) / G;
    const int beg = (int)threadIdx.x / RB * per, end = min(nchunks, beg + per);
    const float* p = partial + std::min<int64_t>(r0 + threadIdx.x % RB, M - 1);
    float sum = 0.f;
    for (int c = beg; c < end; c += U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load(p + min(c + u, end - 1) * mpad);
        sum += pair_sum<U>([&](int u) { return c + u < end ? v[u] : 0.f; });
    }
    if constexpr (G > 1) {
        __shared__ float s_group[NT];
        s_group[threadIdx.x] = sum;
        __syncthreads();
        sum = pair_sum<G>([&](int g) { return s_group[g * RB + threadIdx.x % RB]; });
    }
    return sum;
}

// Column-major A, any shape: a workgroup owns RB = 4 * LR rows (LR lanes of a
// wavefront along the rows, 4 consecutive rows and one 128-bit load per column
// each; its 64 / LR lane groups and 4 wavefronts take interleaved columns) of
// one chunk of columns, U loads in flight per lane.  The last rows' lanes are
// moved back inside A (lanes that own a row twice hold the same sum), and the
// columns past the chunk are clamped and zeroed, so no load is guarded.  The
// scheduling barrier keeps every load of a round ahead of its FMAs: without
// it the compiler consumed each as it came (9003 x 6001: 84 us instead of
// 35).  Four accumulator sets (a lane's u-th column of a round goes to set u
// % 4) keep each FP32 running sum short.  The launcher makes about one
// workgroup per CU: fewer, longer column streams keep HBM pages open.
// Workgroups of one XCD take neighbouring row blocks of a chunk, which share
// the lines at their borders when columns do not start on lines.
// Bound by HBM: 9003 x 6001 (216 MB, columns 4-byte aligned) 45 us with a
// scalar loop over the last partial round and separate row guards, 35 us
// (6.2 TB/s) so.
// STREAM: A is read with the non-temporal hint.
// TINY: fewer than 4 rows, loaded one by one (the last one repeated).
// Chunks' sums of a row block are added in a fixed order by its last workgroup
// to arrive (count: the stream's arrival counters), or by
// sgemv_col_combine_kernel where there are none.
template <int LR, int U, bool STREAM, bool TINY = false>
__global__ __launch_bounds__(NT) void sgemv_col_kernel(int64_t M, int64_t N, float alpha,
                                                       const float* __restrict__ A, int64_t lda,
                                                       const float* __restrict__ x, float beta,
                                                       float* __restrict__ y, float* partial,
                                                       int64_t mpad, int nrb, int nchunks,
                                                       int64_t cols_per_chunk, unsigned* count) {
    constexpr int CG = 64 / LR, STEP = 4 * CG, RB = 4 * LR;
    const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
    const int rb = (int)(b % (unsigned)nrb), ch = (int)(b / (unsigned)nrb);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cg = lane / LR;
    const int64_t r0 = (int64_t)rb * RB;
    const int64_t r = TINY ? 0 : std::min<int64_t>(r0 + 4 * (lane % LR), M - 4);
    const int64_t c0 = ch * cols_per_chunk, c1 = std::min<int64_t>(N, c0 + cols_per_chunk);
    const float* ap = A + r;
    float acc[4][4] = {};
    auto load = [&](int64_t col) {
        const float* p = ap + col * lda;
        if constexpr (TINY) return make_float4(p[0], p[M > 1 ? 1 : 0], p[M - 1], 0.f);
        else return STREAM ? ld4u_nt(p) : ld4u(p);
    };
    auto add = [&](const float4 (&av)[U], const float (&xv)[U]) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float* a = acc[u & 3];
            a[0] = fmaf(av[u].x, xv[u], a[0]);
            a[1] = fmaf(av[u].y, xv[u], a[1]);
            a[2] = fmaf(av[u].z, xv[u], a[2]);
            a[3] = fmaf(av[u].w, xv[u], a[3]);
        }
    };
    int64_t jr = c0;  // first column of the round
    for (; jr + STEP * U <= c1; jr += STEP * U) {
        const int64_t j = jr + wave * CG + cg;
        float4 av[U];
        float xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            xv[u] = x[j + STEP * u];
            av[u] = load(j + STEP * u);
        }
        add(av, xv);
    }
    if (jr < c1) {
        const int64_t j = jr + wave * CG + cg;
        float4 av[U];
        float xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t c = std::min<int64_t>(j + STEP * u, c1 - 1);
            xv[u] = x[c];
            av[u] = load(c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + STEP * u >= c1) {
                xv[u] = 0.f;
                av[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        add(av, xv);
    }
    // Lane sums -> LDS, added in pairs.
    __shared__ float red[STEP][RB];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (r + e >= r0)
            red[wave * CG + cg][r - r0 + e] = (acc[0][e] + acc[1][e]) + (acc[2][e] + acc[3][e]);
    __syncthreads();
    const int t = threadIdx.x;
    const int64_t row = r0 + t;
    const bool mine = t < RB && row < M;
    float sum = 0.f;
    if (mine) sum = pair_sum<STEP>([&](int q) { return red[q][t]; });
    if (nchunks > 1) {
        if (mine) {
            if (count) agent_store(&partial[ch * mpad + row], sum);
            else partial[ch * mpad + row] = sum;
        }
        if (!count || !last_arrival(count + rb * kArrivalStride, (unsigned)nchunks)) return;
        sum = col_chunk_sum<RB>(r0, M, partial, mpad, nchunks,
                                [](const float* p) { return agent_load(p); });
    }
    if (mine) y[row] = beta != 0.f ? alpha * sum + beta * y[row] : alpha * sum;
}

// Column-major A in one pass, for M a multiple of 64 with at least one
// 64-row block per CU and N a multiple of 256 (no partial round, no row
// guard: both measurably slow the loop).  Lane l of a wavefront owns rows
// r0 + 4*(l % 16) .. +3 of column group l / 16, so one load instruction reads
// 4 columns of 64 rows (256 bytes each); wavefront w takes column groups
// 4w .. 4w+3 of every 16 columns, 16 rounds in flight.  Each lane keeps
// four accumulator sets (its u-th column of a round goes to set u % 4),
// added in order; then the 16 lane sums of a row are added in LDS in
// (wavefront, group) order.  Measured 0.91-0.92 of HBM peak at 16384^2.
constexpr int R64_UNROLL = 16;
__global__ __launch_bounds__(NT) void sgemv_col_rows64_kernel(int64_t M, int64_t N, float alpha,
                                                              const float* __restrict__ A,
                                                              int64_t lda,
                                                              const float* __restrict__ x,
                                                              float beta,
                                                              float* __restrict__ y) {
    constexpr int STEP = 16;  // columns per round of the 4 wavefronts
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rq = lane & 15, cg = lane >> 4;
    const int64_t r = (int64_t)blockIdx.x * 64 + 4 * rq;
    const float* ap = A + r;
    float acc[4][4] = {};
    for (int64_t j = wave * 4 + cg; j + STEP * (R64_UNROLL - 1) < N; j += STEP * R64_UNROLL) {
        float4 av[R64_UNROLL];
        float xv[R64_UNROLL];
#pragma unroll
        for (int u = 0; u < R64_UNROLL; ++u) {
            xv[u] = x[j + STEP * u];
            av[u] = ld4u_nt(ap + (j + STEP * u) * lda);
        }
#pragma unroll
        for (int u = 0; u < R64_UNROLL; ++u) {
            float* a = acc[u & 3];
            a[0] = fmaf(av[u].x, xv[u], a[0]);
            a[1] = fmaf(av[u].y, xv[u], a[1]);
            a[2] = fmaf(av[u].z, xv[u], a[2]);
            a[3] = fmaf(av[u].w, xv[u], a[3]);
        }
    }
    __shared__ float red[4][4][64];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        red[wave][cg][4 * rq + e] = ((acc[0][e] + acc[1][e]) + acc[2][e]) + acc[3][e];
    __syncthreads();
    if (threadIdx.x < 64) {
        const int t = threadIdx.x;
        float sum = red[0][0][t];
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (w != 0 || g != 0) sum += red[w][g][t];
        const int64_t row = (int64_t)blockIdx.x * 64 + t;
        float out = alpha * sum;
        if (beta != 0.f) out += beta * y[row];
        y[row] = out;
    }
}

// y = alpha * (sum over the chunks' partials) + beta * y, one row block of
// sgemv_col_kernel per workgroup, in the same order.
template <int RB>
__global__ __launch_bounds__(NT) void sgemv_col_combine_kernel(int64_t M, float alpha,
                                                               const float* __restrict__ partial,
                                                               int64_t mpad, int nchunks,
                                                               float beta, float* __restrict__ y) {
    const int64_t r0 = (int64_t)blockIdx.x * RB, row = r0 + threadIdx.x;
    const float sum = col_chunk_sum<RB>(r0, M, partial, mpad, nchunks,
                                        [](const float* p) { return *p; });
    if (threadIdx.x < RB && row < M)
        y[row] = beta != 0.f ? alpha * sum + beta * y[row] : alpha * sum;
}

// Rows up to which 64-row blocks are used instead of 256-row ones: fewer row
// blocks would leave as many chunks as CUs to add per row (100 x 14000: 55 us
// with 219 chunks added by one thread per row).
constexpr int64_t kColNarrow = 1024;
// Tall matrices of at most 256 columns are read with the non-temporal hint from here
// on (163474 x 64, 42 MB: 7.8 us without, 6.5 with; x 50, 33 MB: 5.0 and 5.8).
constexpr int64_t kTallStreamBytes = (int64_t)40 << 20;

template <int LR, int U, bool STREAM, bool TINY = false>
omb_status launch_col(int64_t M, int64_t N, float alpha, const float* A, int64_t lda,
                      const float* x, float beta, float* y, hipStream_t s) {
    constexpr int RB = 4 * LR, QUANTUM = 4 * (64 / LR) * U;  // rows; columns of one round
    const int64_t nrb = ceil_div(M, RB), cus = device_cu_count();
    if (nrb > 0x7fffffffLL) {
        set_error("sgemv: too many row blocks");
        return OMB_EUNSUPPORTED;
    }
    // At most one workgroup per CU (a few more are a second round for some:
    // 5000 x 12000 with 260 took 48.4 us), chunks of whole rounds.
    const int64_t want = std::max<int64_t>(1, cus / nrb);
    const int64_t rounds = ceil_div(N, QUANTUM);
    const int64_t cpc = ceil_div(rounds, std::min(want, rounds)) * QUANTUM;
    const int64_t nchunks = ceil_div(N, cpc);
    const int64_t mpad = round_up(M, 4);
    Workspace* ws = nullptr;
    OMB_TRY(get_workspace(s, nchunks > 1 ? (size_t)(nchunks * mpad) * sizeof(float) : 0, &ws));
    float* part = reinterpret_cast<float*>(ws->buf);
    unsigned* count = nchunks > 1 && nrb <= kArrivalCounters ? eager_arrivals(s, *ws) : nullptr;
    hipLaunchKernelGGL((sgemv_col_kernel<LR, U, STREAM, TINY>), dim3((unsigned)(nrb * nchunks)),
                       dim3(NT), 0, s, M, N, alpha, A, lda, x, beta, y, part, mpad, (int)nrb,
                       (int)nchunks, cpc, count);
    if (nchunks > 1 && !count)
        hipLaunchKernelGGL(sgemv_col_combine_kernel<RB>, dim3((unsigned)nrb), dim3(NT), 0, s, M,
                           alpha, part, mpad, (int)nchunks, beta, y);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

}  // namespace

// Rows of up to this many columns take 4 rows x 2 loads per wavefront (more
// loads per row would be past its end: 16000 x 600 9.6 us with 2 x 8, 8.7 us).
constexpr int64_t kRowShort = 1024;
// From this many columns on, few rows (up to two wavefronts per CU) are chains of
// rounds: 8 loads per row without the barrier, so that rounds overlap, with addresses
// of their own (1 x 34882 9.4 us with 4 x BATCH, 7.8 with 8, 5.9 so; 300 x 12000 5.7
// and 5.5; but 8 x 8000 4.4 and 4.8, 1000 x 12000 8.9 and 10.0).
constexpr int64_t kRowLong = 10240;

omb_status launch_sgemv_row(int64_t M, int64_t N, float alpha, const float* A, int64_t lda,
                            const float* x, float beta, float* y, hipStream_t s) {
    if (M <= 0) return OMB_OK;
    const int64_t cus = device_cu_count();
    const int64_t waves_per_wg = NT / 64;
    // Tall matrices whose rows start on lines: 16 rows x 1 load, one workgroup
    // per CU (16384^2: 153.4 us, 7.0 TB/s; 8 rows 160).  Rows that do not:
    // 16384 x 9001 took 101 us so, 87.7 with 2 rows x 8 loads in batches.
    // Otherwise batches over 2 rows, or over one where 2 would leave fewer than
    // 3 workgroups per CU (5000 x 12000: 42.1 and 39.8 us), of 8 loads per row
    // where A streams from memory and of 4 where it may be cached, since a
    // shorter batch wastes less of a row's last round (6000 x 4001: 17.1 and
    // 15.9 us).  Before: 4 rows x 4 loads, consumed as they came (50.5 us for
    // 5000 x 12000, 43.1 -> 35.4 for 9003 x 6001, 20.9 for 6000 x 4001).
    const int64_t tall = 16 * waves_per_wg * cus;
    const bool stream = M * N * (int64_t)sizeof(float) > kStreamBytes;
    auto launch = [&](auto kernel, int rows, int64_t most) {
        const int64_t blocks = std::min<int64_t>(ceil_div(ceil_div(M, rows), waves_per_wg), most);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(NT), 0, s, M, N, alpha, A, lda, x,
                           beta, y);
    };
    if (N >= kGemvOff32Cols) {
        if (M >= tall) launch(sgemv_row_kernel<16, 1, true, false, false>, 16, cus);
        else launch(sgemv_row_kernel<1, 8, true, false, true>, 1, 4 * cus);
    } else if (M >= tall && lda % kLineFloats == 0) {
        launch(sgemv_row_kernel<16, 1, true, true, false>, 16, cus);
    } else if (N <= kRowShort) {
        launch(sgemv_row_kernel<4, 2, false, true, true>, 4, 4 * cus);
    } else if (M <= 2 * cus && N > kRowLong && !stream) {
        launch(sgemv_row_kernel<1, 8, false, false, false>, 1, 4 * cus);
    } else if (M < 6 * waves_per_wg * cus) {
        launch(stream ? sgemv_row_kernel<1, 8, true, true, true>
                      : sgemv_row_kernel<1, 4, false, true, true>, 1, 4 * cus);
    } else {
        launch(stream ? sgemv_row_kernel<2, 8, true, true, true>
                      : sgemv_row_kernel<2, 4, false, true, true>, 2, 4 * cus);
    }
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

omb_status launch_sgemv_col(int64_t M, int64_t N, float alpha, const float* A, int64_t lda,
                            const float* x, float beta, float* y, hipStream_t s) {
    if (M <= 0) return OMB_OK;
    const int64_t cus = device_cu_count();
    if (M % 64 == 0 && M / 64 >= cus && N > 0 && N % 256 == 0 && M / 64 <= 0x7fffffffLL) {
        hipLaunchKernelGGL(sgemv_col_rows64_kernel, dim3((unsigned)(M / 64)), dim3(NT), 0, s, M,
                           N, alpha, A, lda, x, beta, y);
        OMB_HIP_TRY(hipGetLastError());
        return OMB_OK;
    }
    if (M < 4) return launch_col<1, 4, false, true>(M, N, alpha, A, lda, x, beta, y, s);
    // Few columns: no more loads in flight per lane than they give one (64 / LR
    // lane groups of 4 wavefronts take columns apart), since the clamped rest cost
    // as much as the others: 400000 x 1 10.0 us with 16, 3.7 so.  The sums are the
    // same for any number of loads.
    const int64_t bytes = M * N * (int64_t)sizeof(float);
    const std::true_type stream;
    const std::false_type cached;
    auto launch = [&](auto lanes, auto loads, auto hint) {
        return launch_col<decltype(lanes)::value, decltype(loads)::value, decltype(hint)::value>(
            M, N, alpha, A, lda, x, beta, y, s);
    };
    const std::integral_constant<int, 1> l1;
    const std::integral_constant<int, 2> l2;
    const std::integral_constant<int, 4> l4;
    const std::integral_constant<int, 8> l8;
    const std::integral_constant<int, 16> l16;
    const std::integral_constant<int, 64> l64;
    if (M <= kColNarrow) {
        if (N <= 16) return launch(l16, l1, cached);
        if (N <= 32) return launch(l16, l2, cached);
        return N <= 64 ? launch(l16, l4, cached) : launch(l16, l8, cached);
    }
    if (N <= 4) return bytes <= kTallStreamBytes ? launch(l64, l1, cached) : launch(l64, l1, stream);
    // Tall ones have more workgroups than CUs, of one chunk: several resident on a CU
    // hide the loads better than more of them per lane (3000000 x 33: 92.8 us with
    // 16, 66.7 with 4).
    if (N <= 256 && ceil_div(M, (int64_t)256) >= cus) {
        if (N <= 128)
            return bytes <= kTallStreamBytes ? launch(l64, l4, cached) : launch(l64, l4, stream);
        return bytes <= kTallStreamBytes ? launch(l64, l8, cached) : launch(l64, l8, stream);
    }
    if (N <= 16) return launch(l64, l4, cached);
    if (N <= 32) return launch(l64, l8, cached);
    return bytes <= kStreamBytes ? launch(l64, l16, cached) : launch(l64, l16, stream);
}

}  // namespace omb
