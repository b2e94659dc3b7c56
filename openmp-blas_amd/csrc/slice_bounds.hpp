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

// The slices that unguarded loads may take of a range of `len` k of a product
// that has `after` more k behind the range, given the larger tail of its two
// operands.  The tail counts from the end of K, not of the range: with K = 129 the
// last three k begin in the block of 128 before the last.  (As a lower bound of
// two ends, min(len, len + after - tail), the same cost products of a partial slice
// up to 2%: 1000 x 700 x 100 9.44 us, 9.30 so.)
template <typename T, typename U>
__host__ __device__ __forceinline__ T full_slices(T len, U after, int tail) {
    const T n = len - (after < tail ? tail - (int)after : 0);
    return n > 0 ? n / kSliceK : 0;
}

}  // namespace omb
