// A 64 x 64 tile of a split-precision product, straight from the FP32 operands:
// the k loop of the grouped items.
//
// 256 threads (4 wavefronts, 32 x 32 of C each) convert 64 lines of A and 64 of
// B^T per 16-k slice and stage the pieces in two LDS buffers; slices are loaded
// up to four ahead in four register sets, one barrier per slice.  What bounds it is the
// conversion (8 values of about 8 operations per thread and slice, against 6 MFMAs of
// 32 cycles per wavefront) and, with few workgroups, a slice's latency.  4096 grouped
// GEMMs of 16 to 512 took 577 us (FP16 pieces: 843) with each slice loaded after the
// one before was consumed and two barriers a slice, 490 (711) so.
#pragma once

#include <algorithm>
#include <type_traits>

#include "split_common.hpp"

namespace omb {
namespace split {

constexpr int kLines = 64;  // lines (rows of A, columns of B) of a tile

// A thread's 4 values per slice of one operand: 4 consecutive k of one line.
// KC: k is the unit stride (4 adjacent threads read 64 bytes of a line), else the
// line is (64 adjacent threads read 256 bytes of each of 4 k).  Lines past the
// operand repeat its last one: what they give is never stored.
template <bool KC, typename P>
struct Quad {
    P p;
    int64_t ld;
    int line, q;

    __device__ __forceinline__ void init(P X, int64_t ld_, int64_t e0, int64_t lines, int tid) {
        ld = ld_;
        line = KC ? tid >> 2 : tid & 63;
        q = KC ? tid & 3 : tid >> 6;
        const int64_t a = std::min<int64_t>(e0 + line, lines - 1);
        p = X + (KC ? a * ld + 4 * q : a + 4 * q * ld);
    }
    __device__ __forceinline__ void load(float (&v)[4], int64_t k0) const {
        if constexpr (KC) {
            const float4 t = ld4u(p + k0);
            v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = p[(k0 + e) * ld];
        }
    }
    // The first kn k of the slice at k0, zeros past them.
    __device__ __forceinline__ void load_tail(float (&v)[4], int64_t k0, int kn) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = 4 * q + e;
            const int64_t d = k < kn ? k0 + e : k0 - 4 * q;  // the slice's first k is valid
            const float t = p[KC ? d : d * ld];
            v[e] = k < kn ? t : 0.f;
        }
    }
};

// The values' pieces (bf16: 2 or 3 planes; f16: two pieces of v * 2^e) into one
// operand's planes of a staged slice.
template <int PL, bool F16>
__device__ __forceinline__ void put_quad(uint4* planes, int line, int q, const float (&v)[4], int e) {
    u16x4 h[PL];
    if constexpr (F16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            _Float16 a, b;
            split2_f16(ldexpf(v[i], e), a, b);
            h[0][i] = __builtin_bit_cast(unsigned short, a);
            h[1][i] = __builtin_bit_cast(unsigned short, b);
        }
    } else {
        split3x4<PL>(v, h);
    }
    uint2* l2 = reinterpret_cast<uint2*>(planes);
#pragma unroll
    for (int pl = 0; pl < PL; ++pl)
        l2[2 * (pl * 2 * kLines + lds_chunk(line, q >> 1)) + (q & 1)] =
            __builtin_bit_cast(uint2, h[pl]);
}

template <int NPROD, bool F16>
struct Staged {  // one slice of both operands
    static constexpr int PL = NPROD == 6 ? 3 : 2;
    static_assert(!F16 || PL == 2, "the FP16 split has two pieces");
    uint4 a[PL * 2 * kLines], b[PL * 2 * kLines];
};

// The sums of a tile over all of K.  G groups of 256 threads take the 256-k
// accumulation blocks in turn (group g: g, g + G, ...); after every G blocks their
// sums meet in LDS (`sum`, G x 2 x 256 float4, two passes) and are added in block
// order, so for any G the bits are those of one group that folds every 256 k.
// out: with one group the 16 sums of each lane; else its group's 16 / G of them
// (values g * 16 / G ..).  Every thread of the workgroup takes every barrier.
template <int NPROD, bool F16, int G, typename QA, typename QB>
__device__ __forceinline__ void tile_sums(const QA& qa, const QB& qb, int ea, int eb, int64_t K,
                                          int group, int tid, Staged<NPROD, F16>* st, float4* sum,
                                          float (&out)[16 / G]) {
    using V = std::conditional_t<F16, f16x8, bf16x8>;
    constexpr int PL = Staged<NPROD, F16>::PL;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1, frow = lane & 31, fh = lane >> 5;
    f32x16 inner[1][1];
    inner[0][0] = f32x16{};
#pragma unroll
    for (int i = 0; i < 16 / G; ++i) out[i] = 0.f;

    const int64_t nfull = K / TK;  // full slices, and k of a partial one
    const int tail = (int)(K - nfull * TK);
    const int64_t blocks = ceil_div(K, (int64_t)TK * kFoldSlices), rounds = ceil_div(blocks, (int64_t)G);
    // This group's j-th slice.
    auto slice = [&](int64_t j) {
        return ((j / kFoldSlices) * G + group) * kFoldSlices + j % kFoldSlices;
    };
    float va[4][4], vb[4][4];  // the slices in flight: slice j in set j % 4
    V fa[PL][1], fb[PL][1];    // fragments of one slice
    auto load = [&](int set, int64_t j) {
        const int64_t k0 = std::min(slice(j), nfull - 1) * TK;
        qa.load(va[set], k0);
        qb.load(vb[set], k0);
    };
    auto put_a = [&](int buf, int set) { put_quad<PL, F16>(st[buf].a, qa.line, qa.q, va[set], ea); };
    auto put_b = [&](int buf, int set) { put_quad<PL, F16>(st[buf].b, qb.line, qb.q, vb[set], eb); };
    auto fragments = [&](int buf) {
        read_frags<PL, 1, 1, kLines, kLines, V, PL>(st[buf].a, wm * 32, wn * 32, frow, fh, fa, fb);
    };
    auto products = [&] { mfma_frags<NPROD, PL, 1, 1, V>(fa, fb, inner); };
    auto fold = [&](int64_t round) {
        if constexpr (G == 1) {
#pragma unroll
            for (int r = 0; r < 16; ++r) out[r] += inner[0][0][r];
        } else {
            const int in_round = (int)std::min<int64_t>(G, blocks - round * G);
            constexpr int OWN = 4 / G;  // float4 of the lane's four added by its group
#pragma unroll
            for (int ps = 0; ps < 2; ++ps) {  // float4 0, 1 of each lane, then 2, 3
                if (group < in_round) {
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int r = 4 * (2 * ps + s);
                        sum[(group * 2 + s) * 256 + tid] =
                            make_float4(inner[0][0][r], inner[0][0][r + 1], inner[0][0][r + 2],
                                        inner[0][0][r + 3]);
                    }
                }
                __syncthreads();
                if (group * OWN / 2 == ps) {
                    for (int w = 0; w < in_round; ++w)
#pragma unroll
                        for (int o = 0; o < OWN; ++o) {
                            const float4 v = sum[(w * 2 + (group * OWN + o) % 2) * 256 + tid];
                            out[4 * o] += v.x;
                            out[4 * o + 1] += v.y;
                            out[4 * o + 2] += v.z;
                            out[4 * o + 3] += v.w;
                        }
                }
                __syncthreads();
            }
        }
        inner[0][0] = f32x16{};
    };
    // Step j (J = j % 4): slice j's fragments are in registers, slice j + 1 in its
    // buffer, slices j + 2 .. j + 4 in flight.  The products of slice j run while
    // slice j + 2 is converted; its buffer was slice j's, read in the step before.
    auto step = [&](int64_t j, auto J) {
        constexpr int S = decltype(J)::value;
        load((S + 1) & 3, j + 5);
        __builtin_amdgcn_sched_barrier(0);
        products();
        put_a(S & 1, (S + 2) & 3);
        fragments((S + 1) & 1);
        put_b(S & 1, (S + 2) & 3);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, 0> s0;
    const std::integral_constant<int, 1> s1;
    const std::integral_constant<int, 2> s2;
    const std::integral_constant<int, 3> s3;
    if (nfull > 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s) load(s, s);
        put_a(0, 0);
        put_b(0, 0);
        load(0, 4);
        put_a(1, 1);
        put_b(1, 1);
        __syncthreads();
        fragments(0);
        __syncthreads();
    }
    for (int64_t r = 0; r < rounds; ++r) {
        // The steps of the round, and those in which this group has a slice.
        const int64_t first = r * G * kFoldSlices;
        auto limit = [&](int64_t s) {
            return (int)std::min<int64_t>(std::max<int64_t>(nfull - s, 0), kFoldSlices);
        };
        const int steps = limit(first), mine = limit(first + group * kFoldSlices);
        const int64_t j0 = r * kFoldSlices;
        int i = 0;
        for (; i + 3 < mine; i += 4) {
            step(j0 + i, s0);
            step(j0 + i + 1, s1);
            step(j0 + i + 2, s2);
            step(j0 + i + 3, s3);
        }
        if (i < mine) {
            step(j0 + i, s0);
            if (i + 1 < mine) step(j0 + i + 1, s1);
            if (i + 2 < mine) step(j0 + i + 2, s2);
            i = mine;
        }
        for (; i < steps; ++i) __syncthreads();
        if (r + 1 < rounds) fold(r);
    }
    if (tail) {
        const bool owner = (blocks - 1) % G == group;
        if (owner) {
            qa.load_tail(va[0], nfull * TK, tail);
            qb.load_tail(vb[0], nfull * TK, tail);
            put_a(0, 0);
            put_b(0, 0);
        }
        __syncthreads();
        if (owner) {
            fragments(0);
            products();
        }
    }
    fold(rounds - 1);
}

// C = alpha * v + beta * C for values r0 .. r0 + NV - 1 of each lane's 16 (the
// 32 x 32 MFMA layout: column lane % 32, row 8*(r/4) + 4*(lane/32) + r%4), C's
// reads ahead of the writes.  em, en (scaled FP16 pieces): the exponents by which
// the tile's rows and columns were scaled, from its first ones on; v is scaled
// back by 2^-(em + en), exactly unless the result leaves FP32's normal range.
template <int NV, typename PC, typename PE>
__device__ __forceinline__ void store_sums(const float (&v)[NV], int r0, int wm, int wn, int lane,
                                           PC C, int64_t ldc, int rows, int cols, float alpha,
                                           float beta, PE em, PE en) {
    const int n = wn * 32 + (lane & 31), m0 = wm * 32 + 4 * (lane >> 5);
    if (n >= cols) return;
    auto row = [&](int i) { return m0 + 8 * ((r0 + i) >> 2) + ((r0 + i) & 3); };
    float old[NV];
    if (beta != 0.f) {
#pragma unroll
        for (int i = 0; i < NV; ++i) old[i] = C[std::min(row(i), rows - 1) * ldc + n];
    }
    const int e = en ? en[n] : 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int m = row(i);
        if (m >= rows) continue;
        const float x = alpha * (en ? ldexpf(v[i], -(em[m] + e)) : v[i]);
        C[m * ldc + n] = beta != 0.f ? x + beta * old[i] : x;
    }
}

}  // namespace split
}  // namespace omb
