// Which 128-bit loads of a plain product's 16-k slices lie inside their operand:
// used by the kernels' k loops, and on the host by a test that walks every loop's
// loads to the ends of small operands.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace omb {

constexpr int kSliceK = 16;

// An operand's side of a tile: E lines (rows of A or columns of B), n of them
// inside the operand; KC: k is the unit stride and lines are ld floats apart,
// else k steps are.  Float offset of 128-bit load e (0 .. 4 * E - 1) of a slice
// from the slice's first element, its line or quad of lines clamped into the
// operand.
template <int E, bool KC>
__host__ __device__ __forceinline__ int64_t slice_load(int e, int n, int64_t ld) {
    return KC ? std::min(e >> 2, n - 1) * ld + (e & 3) * 4
              : (e / (E / 4)) * ld + std::min(e % (E / 4) * 4, (n - 1) & ~3);
}

// k steps at the operand's end that such a load could read past: the last one,
// or the last three when they are less than 4 floats apart.
template <bool KC>
__host__ __device__ __forceinline__ int slice_tail(int n, int64_t ld) {
    return KC || n % 4 == 0 ? 0 : (ld < 4 ? 3 : 1);
}

// The slices of the range [kb, ke) of a product's K that unguarded loads may
// take, given the larger tail of its two operands.  The tail counts from the end
// of K, not of the range: with K = 129 the last three k begin in the block of 128
// before the last.
__host__ __device__ __forceinline__ int64_t full_slices(int64_t kb, int64_t ke, int64_t K,
                                                        int tail) {
    const int64_t n = std::min(ke, K - tail) - kb;
    return n > 0 ? (int64_t)((uint64_t)n / kSliceK) : 0;
}

}  // namespace omb
