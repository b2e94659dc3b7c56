// Shared pieces of the split-BF16 GEMM kernels: tile sizes, the MFMA, the
// swizzled LDS slice layout and the exact 3-way FP32 -> BF16 split.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace omb {
namespace split {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int TM = 128, TN = 128, TK = 16;  // C tile and k slice of one workgroup
constexpr int NT = 256;                      // threads per workgroup (4 wavefronts)
// Tile rows per L2 group: with 4 (against 8, 6 and 5) split BF16 of 8192^3 took 5408 us
// (5496, 5516, 5544), scaled FP16 3292 (3371, 3409, 3465); 4096^3 and below the same.
// The workgroups of an XCD do not keep in step, and with 4 rows miss its L2 less: split
// BF16 of 8192^3 13 to 15 GB a launch, 15 to 17 with 8.
constexpr int kGroupM = 4;
constexpr int kFoldSlices = 16;              // inner MFMA accumulation spans 256 k

__device__ inline f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ inline f32x16 mfma(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// LDS position (in 16-byte chunks, within one plane) of chunk h (0/1) of
// slice row r: the chunk index is flipped by bits 2 and 3 of the row so that
// the 8 or 16 lanes a ds_read_b128 serves per cycle (rows r..r+15, same h)
// hit distinct banks.
__device__ inline int lds_chunk(int r, int h) {
    return (r << 1) | (h ^ ((r >> 2) & 1) ^ ((r >> 3) & 1));
}

// x = h0 + h1 + h2 exactly for |x| >= 2^-110 and zero (each subtraction is
// exact in FP32); below 2^-110 the last piece rounds to BF16's subnormal
// step, within 2^-134.  A finite x above BF16's largest finite value
// (|x| > 0x1.fep127 rounds to infinity) takes h0 truncated instead, so the
// split stays finite and exact.  An infinite or NaN x gives NaN pieces:
// every output it feeds is NaN.
__device__ inline void split3(float x, __bf16& h0, __bf16& h1, __bf16& h2) {
    h0 = (__bf16)x;
    if (__builtin_isinf((float)h0) && !__builtin_isinf(x))
        h0 = __builtin_bit_cast(__bf16, (unsigned short)(__float_as_uint(x) >> 16));
    const float r1 = x - (float)h0;
    h1 = (__bf16)r1;
    h2 = (__bf16)(r1 - (float)h1);
}

// The same for four values into PL planes, without a branch: with the value limited
// to BF16's finite range h0 is split3's (rounded within the range, truncated past
// it).  An infinite x then leaves an infinite rest, whose own rest is NaN; with two
// planes 0 * x makes the first rest NaN.
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
template <int PL>
__device__ __forceinline__ void split3x4(const float (&v)[4], u16x4 (&h)[PL]) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        float r0 = v[i], r1 = v[i + 1];
#pragma unroll
        for (int pl = 0; pl < PL; ++pl) {
            const f32x2 x = pl == 0 ? f32x2{__builtin_amdgcn_fmed3f(r0, -0x1.fep127f, 0x1.fep127f),
                                            __builtin_amdgcn_fmed3f(r1, -0x1.fep127f, 0x1.fep127f)}
                                    : f32x2{r0, r1};
            const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2));
            h[pl][i] = (unsigned short)u;
            h[pl][i + 1] = (unsigned short)(u >> 16);
            if (pl + 1 < PL) {
                r0 -= __uint_as_float(u << 16);
                r1 -= __uint_as_float(u & 0xffff0000u);
            }
            if (PL == 2 && pl == 0) {
                r0 = fmaf(0.f, v[i], r0);
                r1 = fmaf(0.f, v[i + 1], r1);
            }
        }
    }
}

// Scaled FP16 split (two planes per packed slice): the power-of-two exponent
// that brings a line whose largest magnitude is amax into [2^14, 2^15) (0
// for a zero, infinite or NaN amax), and x * 2^e = h0 + h1 + r with
// h0 = fp16(x 2^e) and h1 = fp16(x 2^e - h0) (the subtraction is exact),
// |r| <= max(2^-22 |x 2^e|, 2^-25): relative to x, or FP16's subnormal step.
__device__ inline int line_exp(float amax) {
    if (!(amax > 0.f) || __builtin_isinf(amax)) return 0;
    return 14 - ilogbf(amax);
}
__device__ inline void split2_f16(float xs, _Float16& h0, _Float16& h1) {
    h0 = (_Float16)xs;
    h1 = (_Float16)(xs - (float)h0);
}

// Fragments of one k slice for one wavefront owning BI x BJ blocks of 32x32
// of C (rows wrow0.., columns wcol0.. of the slice), from the swizzled LDS
// slice (PA rows per A plane, PB per B plane; PLA planes in the A part).
// V is the 8-element operand vector of the MFMA: bf16x8 (BF16 pieces) or
// f16x8 (scaled FP16 pieces).
template <int NPLANES, int BI, int BJ, int PA, int PB, typename V, int PLA>
__device__ __forceinline__ void read_frags(const uint4* slice, int wrow0, int wcol0, int frow,
                                           int fh, V (&a)[NPLANES][BI], V (&b)[NPLANES][BJ]) {
    static_assert(NPLANES <= PLA, "the slice holds every plane the products use");
    const uint4* la = slice;
    const uint4* lb = slice + PLA * 2 * PA;
#pragma unroll
    for (int pl = 0; pl < NPLANES; ++pl) {
#pragma unroll
        for (int i = 0; i < BI; ++i) {
            uint4 va = la[pl * 2 * PA + lds_chunk(wrow0 + i * 32 + frow, fh)];
            a[pl][i] = *reinterpret_cast<const V*>(&va);
        }
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
            uint4 vb = lb[pl * 2 * PB + lds_chunk(wcol0 + j * 32 + frow, fh)];
            b[pl][j] = *reinterpret_cast<const V*>(&vb);
        }
    }
}

// The slice's MFMAs from its fragments, smallest products first, all into
// the inner accumulators (NPROD = 6: all pieces of 3 planes; 3: the three
// largest products of 2 planes).  The clock under load falls with the operands that
// change from one MFMA to the next, so the 6-product order keeps one of them: along
// a row of blocks, turning round at each product, neighbours share A's fragment or
// the accumulators.  (The scheduling barriers let all but MFMAs cross.)  8192^3 and
// 6144^3, random operands: 5482 and 2331 us; along a column of blocks 5681 and 2422,
// round the 2 x 2 blocks 5774 and 2443, block by block 5636 and 2387, the
// compiler's order 5908 and 2472.
template <int NPROD, int NPLANES, int BI, int BJ, typename V>
__device__ __forceinline__ void mfma_frags(const V (&a)[NPLANES][BI], const V (&b)[NPLANES][BJ],
                                           f32x16 (&inner)[BI][BJ]) {
    static_assert(NPLANES == (NPROD == 6 ? 3 : 2), "planes of the products");
    if constexpr (NPROD == 6 && BJ > 1) {
        constexpr int pa[6] = {0, 1, 2, 0, 1, 0}, pb[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int t = 0; t < BJ; ++t) {
                    const int j = q & 1 ? BJ - 1 - t : t;
                    inner[i][j] = mfma(a[pa[q]][i], b[pb[q]][j], inner[i][j]);
                    __builtin_amdgcn_sched_barrier(0x496);  // VALU, SALU, memory, LDS, exp
                }
        return;
    }
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
            if constexpr (NPROD == 6) {
                inner[i][j] = mfma(a[0][i], b[2][j], inner[i][j]);
                inner[i][j] = mfma(a[1][i], b[1][j], inner[i][j]);
                inner[i][j] = mfma(a[2][i], b[0][j], inner[i][j]);
            }
            inner[i][j] = mfma(a[0][i], b[1][j], inner[i][j]);
            inner[i][j] = mfma(a[1][i], b[0][j], inner[i][j]);
            inner[i][j] = mfma(a[0][i], b[0][j], inner[i][j]);
        }
}

// MFMAs of one k slice: its fragment reads, then its MFMAs.
// PLA: planes of the A part of the LDS slice (3, or 2 for the two-plane forms).
template <int NPROD, int BI = 2, int BJ = 2, int PA = TM, int PB = TN, typename V = bf16x8,
          int PLA = 3>
__device__ __forceinline__ void mfma_slice(const uint4* slice, int wrow0, int wcol0, int frow,
                                           int fh, f32x16 (&inner)[BI][BJ]) {
    constexpr int NPLANES = NPROD == 6 ? 3 : 2;
    V a[NPLANES][BI], b[NPLANES][BJ];
    read_frags<NPLANES, BI, BJ, PA, PB, V, PLA>(slice, wrow0, wcol0, frow, fh, a, b);
    mfma_frags<NPROD, NPLANES, BI, BJ, V>(a, b, inner);
}

// outer += inner; inner = 0 (FP32 adds: the running sum over K is rounded
// by the vector ALUs, not inside the MFMA accumulation).
template <int BI, int BJ>
__device__ __forceinline__ void fold(f32x16 (&inner)[BI][BJ], f32x16 (&outer)[BI][BJ]) {
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
            outer[i][j] += inner[i][j];
            inner[i][j] = f32x16{};
        }
}

// C = alpha * acc + beta * C for the wavefront's BI x BJ blocks (row-major C).
// 32x32 accumulator layout: lane l holds column l % 32, value r holds row
// 8*(r/4) + 4*(l/32) + r%4.  EXPS (scaled FP16 operands: row m of A was scaled
// by 2^ea[m], column n of B by 2^eb[n]): acc is first scaled back by
// 2^-(ea[m] + eb[n]), exactly unless the result leaves FP32's normal range (as
// the FP32 product itself would).
// BETA: C is read (beta is not zero).  EDGE: the blocks reach past C's rows or
// columns; reads are then clamped into C and the writes guarded.
// Bound by the latency of C's reads: they (and the exponents') are issued for a row
// of blocks ahead of its writes, since a read after a write to C waits for a round
// trip of its own (64 of them for 2 x 2 blocks).  Whole blocks and C = alpha A B take
// code without the guards and tests of the other forms.  Scaled FP16, beta = 1:
// 2500 x 3001 x 1777 154 us element by element, 126 so; 8192 x 8192 x 1024 835 and
// 505; split BF16: 3000 x 3000 x 500 112 and 84, 8192^3 5862 and 5713.
template <bool EXPS, bool BETA, bool EDGE, int BI, int BJ, typename PC, typename PE>
__device__ __forceinline__ void store_blocks(const f32x16 (&acc)[BI][BJ], int rows, int cols,
                                             int lane, PC c, int64_t ldc, float alpha, float beta,
                                             PE ea, PE eb) {
    const int m0 = 4 * (lane >> 5), n0 = lane & 31;
    auto row = [&](int i, int r) { return i * 32 + 8 * (r >> 2) + (r & 3); };  // from m0 on
    const PC lane_c = c + m0 * ldc + n0;
    int en[BJ];
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
        const int n = n0 + 32 * j;
        en[j] = EXPS ? eb[EDGE ? std::min(n, cols - 1) : n] : 0;
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
        float old[BJ][16];
        int em[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + row(i, r), mc = EDGE ? std::min(m, rows - 1) : m;
            em[r] = EXPS ? ea[mc] : 0;
            if constexpr (BETA) {
#pragma unroll
                for (int j = 0; j < BJ; ++j)
                    old[j][r] = EDGE ? c[mc * ldc + std::min(n0 + 32 * j, cols - 1)]
                                     : lane_c[row(i, r) * ldc + 32 * j];
            }
        }
        if constexpr (BETA || EXPS) __builtin_amdgcn_sched_barrier(0);
        auto put = [&](int r, int j) {
            const float a = EXPS ? ldexpf(acc[i][j][r], -(em[r] + en[j])) : acc[i][j][r];
            const float v = alpha * a;
            lane_c[row(i, r) * ldc + 32 * j] = BETA ? v + beta * old[j][r] : v;
        };
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
            if (EDGE && n0 + 32 * j >= cols) continue;
            if (!EDGE || rows >= BI * 32) {
#pragma unroll
                for (int r = 0; r < 16; ++r) put(r, j);
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (m0 + row(i, r) < rows) put(r, j);
            }
        }
    }
}

template <bool EXPS, int BI, int BJ, typename PC, typename PE>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[BI][BJ], int64_t m_base,
                                           int64_t n_base, int lane, PC C, int64_t ldc,
                                           int64_t M, int64_t N, float alpha, float beta,
                                           PE ea, PE eb) {
    const int rows = __builtin_amdgcn_readfirstlane((int)std::min<int64_t>(M - m_base, BI * 32));
    const int cols = __builtin_amdgcn_readfirstlane((int)std::min<int64_t>(N - n_base, BJ * 32));
    if (rows <= 0 || cols <= 0) return;
    const PC c = C + m_base * ldc + n_base;
    if (EXPS) ea += m_base, eb += n_base;
    auto store = [&](auto with_beta, auto edge) {
        store_blocks<EXPS, decltype(with_beta)::value, decltype(edge)::value>(
            acc, rows, cols, lane, c, ldc, alpha, beta, ea, eb);
    };
    const std::true_type yes;
    const std::false_type no;
    if (rows == BI * 32 && cols == BJ * 32) {
        if (beta != 0.f) store(yes, no);
        else store(no, no);
    } else {
        if (beta != 0.f) store(yes, yes);
        else store(no, yes);
    }
}

}  // namespace split
}  // namespace omb
