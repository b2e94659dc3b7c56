// Split products of small and middle sizes in one launch: 64 x 64 tiles straight
// from the FP32 operands (split_tile.hpp), K shared by the groups of 256 threads of
// a workgroup, instead of a pack launch, a product of 128 x 128 tiles with K split
// over workgroups and a launch that adds its partials.  The scaled FP16 form reads
// the line maxima that a launch before it has taken.  Bound by the launches and, for
// few tiles, by the chain of slices of one; the conversion of every operand element
// once per tile that uses it is what leaves large products to the packed path.
// 200 x 300 x 100 split BF16: 14.2 us packed, 6.9 so; 409 x 208 x 197: 17.0 and 9.1;
// 2591 x 311 x 1760: 54.5 and 35.4 (4 groups); 409 x 208 x 197 scaled FP16: 18.7, 13.3.
#include <algorithm>
#include <cmath>

#include "split_tile.hpp"

namespace omb {
namespace {

using namespace split;


struct TArgs {
    int64_t M, N, K;
    float alpha, beta;
    const float* A;
    int64_t lda;
    const float* B;
    int64_t ldb;
    float* C;
    int64_t ldc;
    const unsigned *amax_a, *amax_b;  // F16: bits of the largest |x| of every line
    unsigned tiles_m, tiles_n;
};

// AKC, BKC: k is the operand's unit stride.  A workgroup of one group may share its
// CU with three others, of two with one, of four has it alone.
template <int NPROD, bool F16, int G, bool AKC, bool BKC>
__global__ __launch_bounds__(NT * G, 4) void sgemm_split_tile_kernel(TArgs p) {
    __shared__ Staged<NPROD, F16> st[G][2];
    __shared__ float4 sum[G > 1 ? G * 2 * NT : 1];
    __shared__ int exps[F16 ? 2 : 1][F16 ? kLines : 1];
    const int group = __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT), tid = threadIdx.x % NT;
    int64_t tm, tn;
    group_tile(xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n), p.tiles_m, p.tiles_n, 8, &tm, &tn);
    const int64_t m0 = tm * kLines, n0 = tn * kLines;
    const int rows = (int)std::min<int64_t>(p.M - m0, kLines);
    const int cols = (int)std::min<int64_t>(p.N - n0, kLines);
    int ea = 0, eb = 0;
    Quad<AKC, const float*> qa;
    Quad<BKC, const float*> qb;
    qa.init(p.A, p.lda, m0, p.M, tid);
    qb.init(p.B, p.ldb, n0, p.N, tid);
    if constexpr (F16) {
        if (threadIdx.x < 2 * kLines) {
            const int i = threadIdx.x % kLines;
            const bool a = threadIdx.x < kLines;
            exps[a ? 0 : 1][i] = line_exp(__uint_as_float(
                a ? p.amax_a[m0 + std::min(i, rows - 1)] : p.amax_b[n0 + std::min(i, cols - 1)]));
        }
        __syncthreads();
        ea = exps[0][qa.line];
        eb = exps[1][qb.line];
    }
    float out[16 / G];
    tile_sums<NPROD, F16, G>(qa, qb, ea, eb, p.K, group, tid, st[group], sum, out);
    const int wave = tid >> 6;
    store_sums(out, group * (16 / G), wave >> 1, wave & 1, tid & 63, p.C + m0 * p.ldc + n0, p.ldc, rows,
               cols, p.alpha, p.beta, F16 ? exps[0] : nullptr, F16 ? exps[F16 ? 1 : 0] : nullptr);
}

template <int NPROD, bool F16, int G>
void launch_tiles(const TArgs& p, bool a_kc, bool b_kc, hipStream_t s) {
    const auto kernel = a_kc ? (b_kc ? sgemm_split_tile_kernel<NPROD, F16, G, true, true>
                                     : sgemm_split_tile_kernel<NPROD, F16, G, true, false>)
                             : (b_kc ? sgemm_split_tile_kernel<NPROD, F16, G, false, true>
                                     : sgemm_split_tile_kernel<NPROD, F16, G, false, false>);
    hipLaunchKernelGGL(kernel, dim3(p.tiles_m * p.tiles_n), dim3(NT * G), 0, s, p);
}

template <int NPROD, bool F16>
void launch_groups(int groups, const TArgs& p, bool a_kc, bool b_kc, hipStream_t s) {
    if (groups == 1) return launch_tiles<NPROD, F16, 1>(p, a_kc, b_kc, s);
    if constexpr (NPROD == 6 || F16)
        if (groups == 2) return launch_tiles<NPROD, F16, 2>(p, a_kc, b_kc, s);
    launch_tiles<NPROD, F16, 4>(p, a_kc, b_kc, s);
}

// Models of the time (us) of the launches of a form, fitted to 1100 products (700 of
// the 3-product BF16 form) with M, N and K from 32 to 6144 (geometrically drawn, up
// to 2e10 flop).  One launch of G groups:
//   fixed + amax * K / 1000 + the longer of
//     a workgroup's slices at `step` and rounds of G blocks at `fold` us each, for
//     every wave of workgroups (4 / G to a CU), and
//     the fullest CU's tiles at `tile` + `slice` a slice each.
struct TileModel {
    int groups;  // 0: not built (never the fastest)
    double fixed, step, fold, slice, tile, amax;
};
// Packed: fixed + the operands' (M + N) K at `pack` us per 10^6 + the waves of 512
// workgroups at `slice` a slice + the partials of a split K at `part` us per 10^6.
struct PackedModel {
    double fixed, pack, slice, part, amax;
    double margin;  // what an estimate of the one launch is raised by in the comparison
};
struct FormModel {
    TileModel tile[3];
    PackedModel packed;
};
constexpr FormModel kForms[3] = {
    // BF16, 6 products: the choice takes 1/1.46 of the packed path's time, the
    // fastest 1/1.48; no product of the 1100 lost.
    {{{1, 3.6, 0.220, 0.0, 0.206, 1.45, 7.8}, {2, 3.2, 0.235, 0.3, 0.233, 2.64, 2.5},
      {4, 0.5, 0.398, 5.2, 0.238, 6.2, 0.0}},
     {9.3, 3.05, 0.937, 2.3, 0.0, 1.1}},
    // BF16, 3 products: 1/1.39, the fastest 1/1.41; 0.3% lost more than 3%.
    {{{1, 4.0, 0.208, 0.0, 0.160, 1.25, 4.7}, {}, {4, 0.9, 0.283, 5.1, 0.191, 5.5, 0.0}},
     {9.5, 2.56, 0.583, 1.92, 0.0, 1.1}},
    // Scaled FP16, with the launch that takes the maxima: 1/1.24, the fastest
    // 1/1.28; 0.5% lost more than 3%.
    {{{1, 8.4, 0.236, 0.0, 0.178, 1.59, 7.0}, {2, 7.2, 0.068, 1.0, 0.196, 2.83, 5.1},
      {4, 5.0, 0.336, 5.5, 0.259, 4.84, 0.0}},
     {14.5, 3.63, 0.572, 1.78, 2.3, 1.2}},
};

}  // namespace

int sgemm_split_tile_groups(int64_t M, int64_t N, int64_t K, int nprod, bool f16) {
    // An exact split of K or none, so that the bits do not depend on the choice;
    // and only what the packed path takes.
    int64_t kchunk = K;
    if (sgemm_split_splits(M, N, K, &kchunk) > 1 && kchunk != TK * kFoldSlices) return 0;
    if (ceil_div(K, (int64_t)2 * TK) > 65535) return 0;
    // Scaled FP16 of more k: faster by 10% in 14 of 185 products, and the model did not
    // tell them from those that it made slower (3698 x 53 x 2062: 48 us packed, 57).
    if (f16 && K > 2000) return 0;
    const int64_t tiles = ceil_div(M, (int64_t)kLines) * ceil_div(N, (int64_t)kLines);
    const FormModel& f = kForms[f16 ? 2 : nprod == 3 ? 1 : 0];
    const double cus = (double)device_cu_count(), slices = (double)ceil_div(K, (int64_t)TK);
    const double blocks = (double)ceil_div(K, (int64_t)TK * kFoldSlices);
    const double big = (double)(ceil_div(M, (int64_t)TM) * ceil_div(N, (int64_t)TN));
    const double splits = big > cus ? 1.0 : std::min(blocks, std::floor(2.0 * cus / big));
    const PackedModel& q = f.packed;
    double best = q.fixed + q.pack * 1e-6 * (double)(M + N) * (double)K + q.amax * 1e-3 * (double)K +
                  std::ceil(big * splits / (2.0 * cus)) * slices / splits * q.slice +
                  (splits > 1.0 ? q.part * 1e-6 * (double)M * (double)N * splits : 0.0);
    int groups = 0;
    for (const TileModel& t : f.tile) {
        if (!t.groups || tiles * split::NT * t.groups >= kLaunchItems) continue;
        const double rounds = std::ceil(blocks / t.groups);
        const double chain = t.groups == 1 ? slices * t.step
                                           : rounds * (std::min(16.0, slices) * t.step + t.fold);
        const double waves = std::ceil((double)tiles * t.groups / (4.0 * cus));
        const double full = std::ceil((double)tiles / cus) * (slices * t.slice + t.tile);
        const double time = q.margin * (t.fixed + t.amax * 1e-3 * (double)K +
                                        std::max(waves * chain, full));
        if (time < best) {
            best = time;
            groups = t.groups;
        }
    }
    return groups;
}

omb_status launch_sgemm_split_tile(int groups, int64_t M, int64_t N, int64_t K, float alpha,
                                   const float* A, int64_t lda, bool a_kc, const float* B,
                                   int64_t ldb, bool b_kc, float beta, float* C, int64_t ldc,
                                   int nprod, const unsigned* amax_a, const unsigned* amax_b,
                                   hipStream_t s) {
    const int64_t tiles_m = ceil_div(M, (int64_t)kLines), tiles_n = ceil_div(N, (int64_t)kLines);
    if (tiles_m * tiles_n * split::NT * groups >= kLaunchItems) {
        set_error("sgemm split: too many tiles for one launch");
        return OMB_EUNSUPPORTED;
    }
    const TArgs p{M, N, K, alpha, beta, A, lda, B, ldb, C, ldc, amax_a, amax_b,
                  (unsigned)tiles_m, (unsigned)tiles_n};
    if (amax_a) launch_groups<3, true>(groups, p, a_kc, b_kc, s);
    else if (nprod == 3) launch_groups<3, false>(groups, p, a_kc, b_kc, s);
    else launch_groups<6, false>(groups, p, a_kc, b_kc, s);
    OMB_HIP_TRY(hipGetLastError());
    return OMB_OK;
}

}  // namespace omb
