// Outer product (rank-1 update) and transpose for gfx950: the bandwidth-bound
// BLAS routines beside SGEMV.
//
// SGER, C += alpha * x * y^T (counterpart of amt::outer_prod_helper,
// include/outer.hpp:15-48, whose simd_loop<OUTER> does c[i] += a[i] * b[j]
// line by line, include/simd_loop.hpp:38-50).  Every element is one fused
// multiply-add, c = fma(alpha * x[i], y[j], c), in whichever storage order C
// has: a workgroup updates one row of C along its unit-stride index with
// 128-bit read-modify-writes.
//
// Transpose, C = A^T (counterpart of amt::transpose_helper,
// include/trans.hpp:23-80, out-of-place and square in-place).  When the
// unit-stride index of A is the same matrix index as that of C the transpose
// is a line copy; otherwise 64x64 tiles go through LDS so that both the
// reads and the writes are coalesced.  Square in-place transposes swap tile
// pairs (i, j) and (j, i) through LDS in one workgroup.  Writes are
// non-temporal.
#include <algorithm>

#include "common.hpp"

namespace omb {
namespace {

constexpr int NT = 256;
constexpr int GER_UNROLL = 4;  // 128-bit groups per thread per step

// 128-bit streaming store of 4 consecutive floats at any 4-byte aligned
// address (non-temporal: measured 5-8% faster than plain stores for these
// read-modify-write and copy streams).
__device__ inline void st4u(float* p, float4 v) {
    f32x4_u t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x4_u*>(p));
}

constexpr int kLine = kLineFloats;
// Floats from p to the next 128-byte line: the head of a row, which is written
// element by element so that the 128-bit groups after it fill whole lines.
// A 1 KB wavefront store that starts inside a line leaves two lines of every
// nine partly written, and each is then merged in memory.
__device__ inline int line_head(const float* p) {
    return (int)((0 - (reinterpret_cast<uintptr_t>(p) >> 2)) & (kLine - 1));
}

// Row of this thread's L threads among the workgroup's NT / L: uniform over a
// wavefront, kept scalar so that row addresses are.
template <int L>
__device__ inline int row_in_group() {
    return L == NT ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / L);
}

template <bool COLSCALE>
__device__ inline float4 update4(float alpha, float ur, float4 w, float4 c) {
    if (COLSCALE)
        return make_float4(fmaf(alpha * w.x, ur, c.x), fmaf(alpha * w.y, ur, c.y),
                           fmaf(alpha * w.z, ur, c.z), fmaf(alpha * w.w, ur, c.w));
    return make_float4(fmaf(ur, w.x, c.x), fmaf(ur, w.y, c.y), fmaf(ur, w.z, c.z),
                       fmaf(ur, w.w, c.w));
}

// Rank-1 update of a row-major view D (R x Cc, rows ld apart): D[r][c] +=
// a(r, c) * b(r, c) with a = alpha * (COLSCALE ? v[c] : u[r]) and b the other
// vector's element, so that the x factor of C += alpha x y^T is the scaled
// one in both storage orders.  L threads (a workgroup, or a wavefront for
// short rows) cover a row with 128-bit groups, from the row's first whole
// line with LINES.  Bound by HBM reads and writes.  10007 x 8191 (rows 4-byte
// aligned): 152 us with groups from the row's first element and 4 workgroups
// per CU striding over the rows, 131 us from the first whole line, 113.5 us
// (5.8 TB/s) with a workgroup per row as well; 16384^2: 381 -> 372 us.
// STREAM: C is read with the non-temporal hint (see kStreamBytes).
template <bool COLSCALE, bool STREAM, int L, bool LINES>
__global__ __launch_bounds__(NT) void ger_kernel(int64_t R, int64_t Cc, float alpha,
                                                 const float* __restrict__ u,
                                                 const float* __restrict__ v, float* D,
                                                 int64_t ld) {
    const int lane = threadIdx.x % L;
    for (int64_t r = (int64_t)blockIdx.x * (NT / L) + row_in_group<L>(); r < R;
         r += (int64_t)gridDim.x * (NT / L)) {
        float* row = D + r * ld;
        const float ur = COLSCALE ? u[r] : alpha * u[r];
        const int head = LINES ? (int)std::min<int64_t>(line_head(row), Cc) : 0;
        const int64_t nq = (Cc - head) >> 2;
        float* body = row + head;
        const float* w0 = v + head;
        // head and tail element of this lane (at most 31 + 3 per row), loaded
        // before the groups so that a short row is one round trip
        const int64_t e = lane < head ? lane : 4 * nq + lane;
        float ce = 0.f, we = 0.f;
        if (LINES && e < Cc) ce = row[e], we = v[e];
        int64_t q = lane;
        for (; q + L * (GER_UNROLL - 1) < nq; q += L * GER_UNROLL) {
            float4 c[GER_UNROLL], w[GER_UNROLL];
#pragma unroll
            for (int k = 0; k < GER_UNROLL; ++k) {
                c[k] = STREAM ? ld4u_nt(body + 4 * (q + L * k)) : ld4u(body + 4 * (q + L * k));
                w[k] = ld4u(w0 + 4 * (q + L * k));
            }
#pragma unroll
            for (int k = 0; k < GER_UNROLL; ++k)
                st4u(body + 4 * (q + L * k), update4<COLSCALE>(alpha, ur, w[k], c[k]));
        }
        for (; q < nq; q += L)
            st4u(body + 4 * q, update4<COLSCALE>(alpha, ur, ld4u(w0 + 4 * q), ld4u(body + 4 * q)));
        if (!LINES && e < Cc) ce = row[e], we = v[e];
        if (e < Cc) row[e] = COLSCALE ? fmaf(alpha * we, ur, ce) : fmaf(ur, we, ce);
    }
}

// D (R x Cc, ldd) = S (R x Cc, lds), both row-major: a line copy, the 128-bit
// groups starting on D's first whole line of each row.  STREAM: S is read
// with the non-temporal hint, only where S's groups start on lines too:
// otherwise neighbouring wavefronts share S's lines, and the hint makes each
// fetch them again.
template <bool STREAM, int L, bool LINES>
__global__ __launch_bounds__(NT) void copy_lines_kernel(int64_t R, int64_t Cc,
                                                        const float* __restrict__ S, int64_t lds,
                                                        float* __restrict__ D, int64_t ldd) {
    const int lane = threadIdx.x % L;
    for (int64_t r = (int64_t)blockIdx.x * (NT / L) + row_in_group<L>(); r < R;
         r += (int64_t)gridDim.x * (NT / L)) {
        float* row = D + r * ldd;
        const int head = LINES ? (int)std::min<int64_t>(line_head(row), Cc) : 0;
        const int64_t nq = (Cc - head) >> 2;
        const float* s = S + r * lds + head;
        float* d = row + head;
        const int64_t e = lane < head ? lane : 4 * nq + lane;  // as in ger_kernel
        float se = 0.f;
        if (LINES && e < Cc) se = S[r * lds + e];
        int64_t q = lane;
        for (; q + L * (GER_UNROLL - 1) < nq; q += L * GER_UNROLL) {
            float4 t[GER_UNROLL];
#pragma unroll
            for (int k = 0; k < GER_UNROLL; ++k)
                t[k] = STREAM ? ld4u_nt(s + 4 * (q + L * k)) : ld4u(s + 4 * (q + L * k));
#pragma unroll
            for (int k = 0; k < GER_UNROLL; ++k) st4u(d + 4 * (q + L * k), t[k]);
        }
        for (; q < nq; q += L) st4u(d + 4 * q, ld4u(s + 4 * q));
        if (!LINES && e < Cc) se = S[r * lds + e];
        if (e < Cc) row[e] = se;
    }
}

constexpr int TT = 64;       // transpose tile edge
constexpr int TPAD = TT + 1;  // LDS row pitch (conflict-free column reads)

// Write the transpose of an LDS tile (rows of S at r0.., columns c0..) into
// D (row-major, ldd, Cc x R): D[c][r] = tile[r - r0][c - c0].
__device__ inline void tile_store_t(const float (*tile)[TPAD], float* D, int64_t ldd, int64_t R,
                                    int64_t Cc, int64_t r0, int64_t c0) {
    const int g = threadIdx.x & 15, cc = threadIdx.x >> 4;
#pragma unroll
    for (int k = 0; k < TT / 16; ++k) {
        const int lc = cc + 16 * k;
        const int64_t c = c0 + lc, r = r0 + 4 * g;
        if (c >= Cc) continue;
        const float4 v = make_float4(tile[4 * g + 0][lc], tile[4 * g + 1][lc],
                                     tile[4 * g + 2][lc], tile[4 * g + 3][lc]);
        float* p = D + c * ldd;
        if (r + 3 < R) {
            st4u(p + r, v);
        } else {
            if (r < R) p[r] = v.x;
            if (r + 1 < R) p[r + 1] = v.y;
            if (r + 2 < R) p[r + 2] = v.z;
        }
    }
}

// The 4 rows of a TT x TT tile of S (row-major, lds) at (r0, c0) that
// thread t reads: 4-float group t % 16 of rows t / 16 + 16k, zero past the
// edges; kept in registers so that several tiles' loads are in flight.
__device__ inline void tile_regs(float4 (&v)[TT / 16], const float* S, int64_t lds, int64_t R,
                                 int64_t Cc, int64_t r0, int64_t c0) {
    const int g = threadIdx.x & 15, rr = threadIdx.x >> 4;
#pragma unroll
    for (int k = 0; k < TT / 16; ++k) {
        const int64_t r = r0 + rr + 16 * k, c = c0 + 4 * g;
        v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < R) {
            if (c + 3 < Cc) {
                v[k] = ld4u_nt(S + r * lds + c);
            } else {
                const float* p = S + r * lds;
                if (c < Cc) v[k].x = p[c];
                if (c + 1 < Cc) v[k].y = p[c + 1];
                if (c + 2 < Cc) v[k].z = p[c + 2];
            }
        }
    }
}

__device__ inline void tile_put(float (*tile)[TPAD], const float4 (&v)[TT / 16]) {
    const int g = threadIdx.x & 15, rr = threadIdx.x >> 4;
#pragma unroll
    for (int k = 0; k < TT / 16; ++k) {
        const int lr = rr + 16 * k;
        tile[lr][4 * g + 0] = v[k].x;
        tile[lr][4 * g + 1] = v[k].y;
        tile[lr][4 * g + 2] = v[k].z;
        tile[lr][4 * g + 3] = v[k].w;
    }
}

// D (Cc x R, ldd) = S^T (S: R x Cc, lds), both row-major: one tile of RT rows
// of S and CT rows of D per workgroup, through LDS.  Each row of D is written
// from its tile's start moved back by the row's offset in its 128-byte line
// (0 .. 31 floats): every 128-bit store then fills whole lines, with a scalar
// guard only at the row's ends.  For that the workgroup reads the 31 rows of
// S before the tile too (none when D's rows start on lines); they are the
// neighbour's rows, and the workgroups of one XCD take neighbouring tiles
// along r, so they come from its L2.  Reads are cached, as tiles share S's
// lines as well.  Bound by HBM.  Measured against 64x64 tiles stored from
// their own start, with a second launch for partial tiles: 8001 x 12007 (rows
// 4-byte aligned; partly written lines are merged in memory) 308 -> 150 us
// (5.1 TB/s), 3001 x 2503 24.7 -> 11.4 us, 4096^2 27.2 -> 21.4 us.
// diag: tiles step along c with r.  With rows 32 KB apart a column of tiles
// reads, and a row of them writes, the same memory channels: 8192^2 118 us
// without, 99 us with it, 16384^2 462 and 412 us; other strides lose 2-9%
// by it (8000 x 12032: 144 and 158 us).
template <int RT, int CT>
__global__ __launch_bounds__(NT) void transpose_lines_kernel(int64_t R, int64_t Cc, unsigned GR,
                                                             unsigned GC,
                                                             const float* __restrict__ S,
                                                             int64_t lds, float* __restrict__ D,
                                                             int64_t ldd, int on_lines, int diag) {
    constexpr int LR = RT + kLine;                      // rows of S held in LDS
    constexpr int CQ = CT / 4, RPI = NT / CQ;           // loads: groups per row, rows per step
    constexpr int RQ = RT / 4, CPI = NT / RQ;           // stores: groups per row of D, rows per step
    static_assert(kLine % RPI == 0 && RT % RPI == 0 && CT % CPI == 0, "whole steps");
    __shared__ float tile[LR][CT + 1];
    const int cq = threadIdx.x % CQ, rr = threadIdx.x / CQ;
    const int g = threadIdx.x % RQ, cc = threadIdx.x / RQ;
    const uint64_t ntiles = (uint64_t)GR * GC;
    // XCD x (workgroups x mod 8) takes tiles [x, x+1) * ntiles / 8, r fastest.
    const unsigned x = blockIdx.x & 7;
    const uint64_t end = ntiles * (x + 1) / 8;
    for (uint64_t t = ntiles * x / 8 + (blockIdx.x >> 3); t < end; t += gridDim.x >> 3) {
        // t < 2^32: a matrix of that many tiles is 32 TB
        const unsigned q = (unsigned)t / GR, gr = (unsigned)t % GR, gc = diag ? (q + gr) % GC : q;
        const int64_t r0 = (int64_t)gr * RT, c0 = (int64_t)gc * CT;
        const bool full = (on_lines || r0 >= kLine) && r0 + RT <= R && c0 + CT <= Cc;
        float4 v[LR / RPI];
        if (full) {
#pragma unroll
            for (int k = 0; k < LR / RPI; ++k)
                if (k * RPI >= kLine || !on_lines)
                    v[k] = ld4u(S + (r0 - kLine + rr + RPI * k) * lds + c0 + 4 * cq);
        } else {  // clamped indices: what lies outside S is not stored
#pragma unroll
            for (int k = 0; k < LR / RPI; ++k) {
                // steps of no row of S at all are left out (65 x 2000000: 321 us with
                // them, 289 so)
                const int64_t first = r0 - kLine + RPI * k;
                if (first >= R || first + RPI <= 0) {
                    v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
                    continue;
                }
                const int64_t r = first + rr, c = c0 + 4 * cq;
                const float* p = S + std::min(std::max<int64_t>(r, 0), R - 1) * lds;
                if (c + 3 < Cc) {
                    v[k] = ld4u(p + c);
                } else {
                    v[k] = make_float4(p[std::min(c, Cc - 1)], p[std::min(c + 1, Cc - 1)],
                                       p[std::min(c + 2, Cc - 1)], 0.f);
                }
            }
        }
        __syncthreads();  // the previous tile has been written out
#pragma unroll
        for (int k = 0; k < LR / RPI; ++k) {
            if (k * RPI < kLine && on_lines) continue;
            float* p = &tile[rr + RPI * k][4 * cq];
            p[0] = v[k].x;
            p[1] = v[k].y;
            p[2] = v[k].z;
            p[3] = v[k].w;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < CT / CPI; ++k) {
            const int lc = cc + CPI * k;
            float* d = D + (c0 + lc) * ldd;
            const int back = (kLine - line_head(d + r0)) & (kLine - 1);
            const int lr = kLine - back + 4 * g;
            const int64_t r = r0 - back + 4 * g;
            const float4 o = make_float4(tile[lr][lc], tile[lr + 1][lc], tile[lr + 2][lc],
                                         tile[lr + 3][lc]);
            if (full) {
                st4u(d + r, o);
            } else if (c0 + lc < Cc) {
                if (r >= 0 && r + 3 < R) {
                    st4u(d + r, o);
                } else {
                    if (r >= 0 && r < R) d[r] = o.x;
                    if (r >= -1 && r + 1 < R) d[r + 1] = o.y;
                    if (r >= -2 && r + 2 < R) d[r + 2] = o.z;
                    if (r >= -3 && r + 3 < R) d[r + 3] = o.w;
                }
            }
        }
    }
}

// The same for thin matrices, which are one row or one column of tiles: 64 x 64
// tiles with guards, one per step.  (µs: this, transpose_lines_kernel.)
//  - R < 64: D's rows are short, and moving them back to lines spreads each over
//    more lanes that store little: 1 x 2000000 26 and 71, 9 x 2000000 39 and 76
//    (176 in its large tiles), 48 x 2000000 129 and 196.
//  - Cc <= 10: few of a tile's columns are there: 2000000 x 1 23 and 30, 300000 x 9
//    6.4 and 7.3, 2000000 x 12 50 and 38.
//  - 32 < Cc < 64 where D's rows start on lines: 2000000 x 40 113 and 175 (where
//    they do not: 227 and 158).
bool thin_transpose(int64_t R, int64_t Cc, bool on_lines) {
    return R < 64 || Cc <= 10 || (on_lines && Cc > 32 && Cc < 64);
}
__global__ __launch_bounds__(NT) void transpose_thin_kernel(int64_t R, int64_t Cc, int64_t ntiles,
                                                            const float* __restrict__ S,
                                                            int64_t lds, float* __restrict__ D,
                                                            int64_t ldd) {
    __shared__ float tile[TT][TPAD];
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int64_t r0 = R < TT ? 0 : t * TT, c0 = R < TT ? t * TT : 0;
        float4 v[TT / 16];
        tile_regs(v, S, lds, R, Cc, r0, c0);
        __syncthreads();  // the previous tile has been written out
        tile_put(tile, v);
        __syncthreads();
        tile_store_t(tile, D, ldd, R, Cc, r0, c0);
    }
}

// Square in-place transpose of A (n x n, row-major view with ld): workgroup
// (bj, bi) with bi <= bj swaps tile (bi, bj) with tile (bj, bi), each
// transposed; bi == bj transposes the diagonal tile.  Workgroups below the
// diagonal have nothing to do.
__global__ __launch_bounds__(NT) void transpose_inplace_kernel(int64_t n, float* A, int64_t ld) {
    __shared__ float t0[TT][TPAD];
    __shared__ float t1[TT][TPAD];
    const int64_t bj = blockIdx.x, bi = blockIdx.y;
    if (bi > bj) return;
    const int64_t r0 = bi * TT, c0 = bj * TT;
    float4 v0[TT / 16], v1[TT / 16];  // both tiles' loads in flight at once
    tile_regs(v0, A, ld, n, n, r0, c0);
    if (bi != bj) tile_regs(v1, A, ld, n, n, c0, r0);
    tile_put(t0, v0);
    if (bi != bj) tile_put(t1, v1);
    __syncthreads();
    tile_store_t(t0, A, ld, n, n, r0, c0);  // (bi, bj)^T -> (bj, bi)
    if (bi != bj) tile_store_t(t1, A, ld, n, n, c0, r0);
}

// Split of the rows for the rank-1 and copy kernels, by what bounds them:
// rows of more than 1024 floats take a workgroup each and start on whole
// lines; shorter ones are bound by the rate workgroups start at and by the
// round trips of a row, so up to 512 floats a wavefront takes each row (outer
// 16382 x 300: 11.3 -> 9.3 us; a workgroup per row 12.8), and between the two
// 4 workgroups per CU stride over the rows (copy of 16000 x 900: 18.8 us; a
// wavefront per row 26, a workgroup per row 19.6).
struct RowSplit {
    bool by_wave, lines;
    unsigned grid;
};
RowSplit row_split(int64_t rows, int64_t Cc) {
    const bool by_wave = Cc <= 512, lines = Cc > 1024;
    const int64_t most = by_wave || lines ? 1 << 22 : 4 * (int64_t)device_cu_count();
    const int64_t groups = by_wave ? ceil_div(rows, NT / 64) : rows;
    return {by_wave, lines, (unsigned)std::max<int64_t>(1, std::min(groups, most))};
}

bool overlaps(const float* a, int64_t na, const float* b, int64_t nb) {
    return na > 0 && nb > 0 && a < b + nb && b < a + na;
}

int64_t span_of(int64_t rows, int64_t cols, int64_t rs, int64_t cs) {
    return (rows <= 0 || cols <= 0) ? 0 : (rows - 1) * rs + (cols - 1) * cs + 1;
}

}  // namespace
}  // namespace omb

using namespace omb;

extern "C" omb_status omb_sger(int64_t M, int64_t N, float alpha, const float* x, const float* y,
                               float* C, int64_t rsC, int64_t csC, omb_stream_t stream) {
    clear_error();
    if (M < 0 || N < 0) {
        set_error("omb_sger: negative size");
        return OMB_EINVAL;
    }
    if (M == 0 || N == 0) return OMB_OK;
    if (!x || !y || !C) {
        set_error("omb_sger: null pointer");
        return OMB_EINVAL;
    }
    bool row = false;
    int64_t ld = 0;
    OMB_TRY(resolve_layout("omb_sger C", M, N, rsC, csC, &row, &ld));
    hipStream_t s = (hipStream_t)stream;
    // row-major C: its rows; column-major C: its columns are the lines, and
    // rows of the view are j
    const int64_t R = row ? M : N, Cc = row ? N : M;
    const bool stream_c = R * Cc > kStreamBytes / (int64_t)sizeof(float);
    const RowSplit sp = row_split(R, Cc);
    const float *u = row ? x : y, *v = row ? y : x;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(sp.grid), dim3(NT), 0, s, R, Cc, alpha, u, v, C, ld);
    };
    if (sp.by_wave && row) launch(ger_kernel<false, false, 64, false>);
    else if (sp.by_wave) launch(ger_kernel<true, false, 64, false>);
    else if (!sp.lines && row) launch(ger_kernel<false, false, NT, false>);
    else if (!sp.lines) launch(ger_kernel<true, false, NT, false>);
    else if (row) launch(stream_c ? ger_kernel<false, true, NT, true> : ger_kernel<false, false, NT, true>);
    else launch(stream_c ? ger_kernel<true, true, NT, true> : ger_kernel<true, false, NT, true>);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

extern "C" omb_status omb_stranspose(int64_t M, int64_t N, const float* A, int64_t rsA,
                                     int64_t csA, float* C, int64_t rsC, int64_t csC,
                                     omb_stream_t stream) {
    clear_error();
    if (M < 0 || N < 0) {
        set_error("omb_stranspose: negative size");
        return OMB_EINVAL;
    }
    if (M == 0 || N == 0) return OMB_OK;
    if (!A || !C) {
        set_error("omb_stranspose: null pointer");
        return OMB_EINVAL;
    }
    bool a_row = false, c_row = false;
    int64_t lda = 0, ldc = 0;
    OMB_TRY(resolve_layout("omb_stranspose A", M, N, rsA, csA, &a_row, &lda));
    OMB_TRY(resolve_layout("omb_stranspose C", N, M, rsC, csC, &c_row, &ldc));
    if (overlaps(A, span_of(M, N, rsA, csA), C, span_of(N, M, rsC, csC))) {
        set_error("omb_stranspose: A and C overlap (use omb_stranspose_inplace)");
        return OMB_EINVAL;
    }
    // Row-major views: S is A as stored (R x Cc), D is C as stored.
    //   A row (M x N), C row (N x M): D = S^T           -> tiles
    //   A row,         C col: C as stored is M x N = S  -> copy
    //   A col (N x M as stored), C row (N x M) = S      -> copy
    //   A col,         C col (M x N as stored) = S^T    -> tiles
    const int64_t R = a_row ? M : N, Cc = a_row ? N : M;
    hipStream_t s = (hipStream_t)stream;
    const bool on_lines = reinterpret_cast<uintptr_t>(C) % (kLine * sizeof(float)) == 0 &&
                          ldc % kLine == 0;
    if (a_row == c_row && thin_transpose(R, Cc, on_lines)) {
        const int64_t ntiles = ceil_div(R < TT ? Cc : R, (int64_t)TT);
        const dim3 grid((unsigned)std::min<int64_t>(ntiles, kLaunchItems / NT / 4));
        hipLaunchKernelGGL(transpose_thin_kernel, grid, dim3(NT), 0, s, R, Cc, ntiles, A, lda, C, ldc);
    } else if (a_row == c_row) {
        const bool diag = on_lines && (lda % 8192 == 0 || ldc % 8192 == 0);
        // (2000000 x 12: 101 us in the large tiles, 38 so; 64 x 300000 36 and 29)
        const bool big = R * Cc >= (int64_t)1 << 24 && R > 64 && Cc > 32;
        const int64_t rt = big ? 128 : 64, ct = big ? 64 : 32;
        // rows of D moved back by up to 31 floats can need one tile more
        const int64_t GR = ceil_div(R + (on_lines ? 0 : kLine - 1), rt), GC = ceil_div(Cc, ct);
        // (the kernel strides over the tiles; 2 x 2^30 has as many as exceed a launch)
        const dim3 grid((unsigned)std::min<int64_t>(round_up(GR * GC, 8), kLaunchItems / NT / 4));
        const auto kernel = big ? transpose_lines_kernel<128, 64> : transpose_lines_kernel<64, 32>;
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, s, R, Cc, (unsigned)GR, (unsigned)GC, A, lda, C, ldc,
                           on_lines ? 1 : 0, diag ? 1 : 0);
    } else {
        // whole-line groups of C are whole-line groups of A on every row
        const bool stream = (reinterpret_cast<uintptr_t>(A) - reinterpret_cast<uintptr_t>(C)) %
                                    (kLine * sizeof(float)) == 0 &&
                            (lda - ldc) % kLine == 0;
        const RowSplit sp = row_split(R, Cc);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(sp.grid), dim3(NT), 0, s, R, Cc, A, lda, C, ldc);
        };
        if (sp.by_wave) launch(copy_lines_kernel<false, 64, false>);
        else if (!sp.lines) launch(copy_lines_kernel<false, NT, false>);
        else launch(stream ? copy_lines_kernel<true, NT, true> : copy_lines_kernel<false, NT, true>);
    }
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

extern "C" omb_status omb_stranspose_inplace(int64_t n, float* A, int64_t ld,
                                             omb_stream_t stream) {
    clear_error();
    if (n < 0 || (n > 0 && ld < n)) {
        set_error("omb_stranspose_inplace: need n >= 0 and ld >= n");
        return OMB_EINVAL;
    }
    if (n == 0) return OMB_OK;
    if (!A) {
        set_error("omb_stranspose_inplace: null pointer");
        return OMB_EINVAL;
    }
    const int64_t t = ceil_div(n, TT);
    if (t > 65535) {
        set_error("omb_stranspose_inplace: matrix too large for one launch");
        return OMB_EUNSUPPORTED;
    }
    hipLaunchKernelGGL(transpose_inplace_kernel, dim3((unsigned)t, (unsigned)t), dim3(NT), 0,
                       (hipStream_t)stream, n, A, ld);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}
