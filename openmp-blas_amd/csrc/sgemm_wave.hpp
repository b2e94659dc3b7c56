// One wavefront's share of a plain FP32 product: its own 16-k slices of A and B
// staged through its own LDS buffer, 4*GR x 4*GC outputs per lane.  Used by the
// kernel that divides K among wavefronts and by the grouped items.
#pragma once

#include <algorithm>

#include "slice_bounds.hpp"

namespace omb {
namespace wave {

constexpr int BK = kSliceK;
constexpr int BLOCK_K = 128;  // k per accumulation block, as sgemm_f32.hip
constexpr int PAD = 4;

template <typename Off>
__device__ __forceinline__ const float* at_bytes(const float* p, Off off) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + off);
}
template <typename Off>
__device__ __forceinline__ gcfloat* at_bytes(gcfloat* p, Off off) {
    typedef const OMB_GLOBAL char gcchar;
    return reinterpret_cast<gcfloat*>(reinterpret_cast<gcchar*>(p) + off);
}

// Orders a wavefront's LDS writes before its other lanes' reads (and the
// reverse): the hardware keeps the order, this keeps the compiler's.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One operand of a wavefront's tile: E rows (of A) or columns (of B^T), called
// lines, starting at line e0; KC: k is the unit stride.  load() brings a full
// slice into registers, load_guarded() a partial one, store() puts it into LDS
// as [k][line].
template <int E, bool KC, typename Off, typename P>
struct WaveSide {
    static constexpr int L = E / 16;  // float4 per lane and slice
    P p;             // line e0 (wavefront-uniform, as is the k of a load: the
                     // loads add a lane's offset to a scalar address)
    int64_t ld;
    int n;           // lines of the operand from e0
    int lane;

    __device__ __forceinline__ void init(P X, int64_t ld_, int64_t e0, int64_t extent,
                                         int lane_) {
        p = X + (KC ? e0 * ld_ : e0);
        ld = ld_;
        n = (int)std::min<int64_t>(extent - e0, E);
        lane = lane_;
    }
    // byte offset of load i: line (KC) or quad of lines, clamped into the operand
    __device__ __forceinline__ Off offset(int i) const {
        return (Off)(4 * slice_load<E, KC>(lane + 64 * i, n, ld));
    }
    __device__ __forceinline__ void load(float4 (&v)[L], const Off (&off)[L], int64_t k0) const {
        const P q = p + (KC ? k0 : k0 * ld);
#pragma unroll
        for (int i = 0; i < L; ++i) v[i] = ld4u(at_bytes(q, off[i]));
    }
    __device__ __forceinline__ int tail() const { return slice_tail<KC>(n, ld); }
    // k0 .. k1-1 are the valid k of the slice (k1 <= K)
    __device__ __forceinline__ void load_guarded(float4 (&v)[L], int64_t k0, int64_t k1) const {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int e = lane + 64 * i;
            float t[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int64_t line = min(KC ? e >> 2 : e % (E / 4) * 4 + c, n - 1);
                const int64_t k = k0 + (KC ? (e & 3) * 4 + c : e / (E / 4));
                const int64_t b = std::min(k, k1 - 1);
                const float x = p[KC ? line * ld + b : b * ld + line];
                t[c] = k < k1 ? x : 0.f;
            }
            v[i] = make_float4(t[0], t[1], t[2], t[3]);
        }
    }
    __device__ __forceinline__ void store(float (*s)[E + PAD], const float4 (&v)[L]) const {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int e = lane + 64 * i;
            if constexpr (KC) {
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
};

template <int GR, int GC>
struct WaveStage {
    float a[BK][32 * GR + PAD], b[BK][32 * GC + PAD];
};

// inner += the staged slice: lane (ly, lx) of 8 x 8 owns rows g*32 + ly*4 + 0..3 and
// columns h*32 + lx*4 + 0..3, each column's sum in place acc_slot of its quad.
template <int GR, int GC>
__device__ __forceinline__ void wave_compute(const WaveStage<GR, GC>& st, int lane,
                                             acc4 (&inner)[4 * GR][GC]) {
    const int lx = lane & 7, ly = lane >> 3;
    float4 fa[2][GR], fb[2][GC];  // fragments of this k and of the next one
    auto fragment = [&](int k, int set) {
#pragma unroll
        for (int g = 0; g < GR; ++g)
            fa[set][g] = *reinterpret_cast<const float4*>(&st.a[k][g * 32 + ly * 4]);
#pragma unroll
        for (int h = 0; h < GC; ++h)
            fb[set][h] = *reinterpret_cast<const float4*>(&st.b[k][h * 32 + lx * 4]);
    };
    fragment(0, 0);
#pragma unroll
    for (int k = 0; k < BK; ++k) {
        if (k + 1 < BK) fragment(k + 1, (k + 1) & 1);
        const float* a = reinterpret_cast<const float*>(fa[k & 1]);
#pragma unroll
        for (int i = 0; i < 4 * GR; ++i)
#pragma unroll
            for (int h = 0; h < GC; ++h) {
                const float4 v = fb[k & 1][h];
                acc4& s = inner[i][h];
                s[acc_slot(0)] = fmaf(a[i], v.x, s[acc_slot(0)]);
                s[acc_slot(1)] = fmaf(a[i], v.y, s[acc_slot(1)]);
                s[acc_slot(2)] = fmaf(a[i], v.z, s[acc_slot(2)]);
                s[acc_slot(3)] = fmaf(a[i], v.w, s[acc_slot(3)]);
            }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Keeps each tuple in four consecutive registers through a loop.
template <int TR, int GC>
__device__ __forceinline__ void pin(acc4 (&inner)[TR][GC]) {
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int h = 0; h < GC; ++h) asm volatile("" : "+v"(inner[i][h]));
}

}  // namespace wave
}  // namespace omb
