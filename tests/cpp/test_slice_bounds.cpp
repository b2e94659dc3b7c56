// Host walk of the plain products' unguarded slice loads (csrc/slice_bounds.hpp):
// over every range of K that a kernel's loop takes (blocks of 128 k, splits of
// several blocks, all of K) each 128-bit load must end inside its operand, and no
// more slices than the end of K asks for may be left to the guarded loads.
// Prints "ok <checks>" or the first load past an operand.
#include <cstdio>
#include <cstdlib>

#include "slice_bounds.hpp"

using namespace omb;

static long g_checks = 0;

// n: lines from e0 on inside the operand; lines at most E: the operand's own extent
template <int E, bool KC>
static void walk(int n, int64_t ld, int64_t K, int64_t range) {
    const int tail = slice_tail<KC>(n, ld);
    const int64_t last = KC ? (n - 1) * ld + K - 1 : (K - 1) * ld + n - 1;
    for (int64_t kb = 0; kb < K; kb += range) {
        const int64_t ke = std::min(K, kb + range), full = full_slices(ke - kb, K - ke, tail);
        bool ok = full >= 0 && kb + full * kSliceK <= ke;
        for (int64_t s = 0; s < full; ++s)
            for (int e = 0; e < 4 * E; ++e) {
                const int64_t k0 = kb + s * kSliceK;
                ok = ok && (KC ? k0 : k0 * ld) + slice_load<E, KC>(e, n, ld) + 3 <= last;
            }
        // whole slices before the tail are not left to the guarded loads
        ok = ok && (std::min(ke, K - tail) - kb < (full + 1) * kSliceK);
        ++g_checks;
        if (!ok) {
            std::fprintf(stderr, "FAILED: E %d kc %d n %d ld %ld K %ld range %ld block %ld\n", E, KC,
                         n, (long)ld, (long)K, (long)range, (long)(kb / range));
            std::exit(1);
        }
    }
}

template <int E>
static void side(int64_t K, int64_t range) {
    const int lines[] = {1, 2, 3, 4, 5, E - 1, E};
    for (int n : lines)
        for (int64_t ld = n; ld <= std::max(n, 4) + 1; ++ld) walk<E, false>(n, ld, K, range);
    for (int n : {1, 3, E}) walk<E, true>(n, K, K, range);
}

int main() {
    for (int64_t K = 1; K <= 1100; ++K) {
        const int64_t off = K % 128;  // every K near a boundary of blocks, some between
        if (off > 20 && off < 108 && K % 7) continue;
        for (int64_t range : {(int64_t)128, (int64_t)256, (int64_t)384, K}) {
            side<32>(K, range);
            side<64>(K, range);
            side<128>(K, range);
        }
    }
    std::printf("ok %ld\n", g_checks);
    return 0;
}
