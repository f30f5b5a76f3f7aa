// Choice and launch of the products on the bf16 matrix cores (the kernels and
// their reasons: ts_hip_gemm_split.h).
#include "ts_hip_gemm_split.h"

namespace tship {

// Products of fewer operations than this stay on the fp32 instructions.  Against
// the fp32 kernels (us, theirs and these): 1024 x 1024 x 784, 1.6e9: 18.6, 21.2;
// 1024 x 1024 x 1024, 2.1e9: 22.9, 22.7; 2000 x 300 x 2000, 2.4e9: 42, 39; NT 640 x
// 640 x 3000, 2.5e9: 65, 45.  Where a size is no multiple of four those load
// element by element: 1000 x 1000 x 500, 1.0e9, aligned: 14.2, 18.5; 999 x 777 x
// 1001, 1.6e9: 44, 24; 1339 x 288 x 2112, 1.6e9: 46, 40.
constexpr double kSplitMinFlop = 2.2e9, kSplitMinFlopRagged = 1.5e9;

// Untransposed products with this many elements of B and more stay there too.
// They are the forward products of wide layers, and a relu unit whose input
// lies within rounding of zero takes either branch by the order of a sum: two
// correct roundings of the forward products of a deep network train apart,
// neither nearer to 64 bits, the more the wider and deeper it is.  Two Adam
// steps of six layers, the largest difference of a weight matrix (2-norm) from
// the fp32 kernels' with the forward products here: width 1024 9e-4, 2048
// 1.3e-3, 2880 1.9e-3, 3328 2.5e-3, 4096 and 4100 4.5e-3, at any batch; with them
// on the fp32 instructions 1.6e-4.  The line keeps the networks past 2e-3 at the
// results that the fp32 kernels give.  It costs 8192 x 4096 x 4096 1850 us instead
// of 1440, 8192 x 4100 x 4096 2840 instead of 1570.
constexpr size_t kSplitForwardMaxB = size_t(1) << 23;

SplitPlan split_plan(int trans_a, int trans_b, size_t M, size_t N, size_t K, size_t batches) {
    SplitPlan p;
    const size_t lim = size_t(1) << 23;
    if (M < 64 || N < 64 || K < 64 || M > lim || N > lim || K > lim || batches == 0) return p;
    if (K * N <= 16384) return p;  // (where ts_hip_gemm_colsum_bsum has its sum in the fp32 tiles' grid)
    if (!trans_a && !trans_b && K * N >= kSplitForwardMaxB) return p;
    const bool ragged = M % 4 != 0 || N % 4 != 0 || K % 4 != 0;
    if (2.0 * M * N * K * batches < (ragged ? kSplitMinFlopRagged : kSplitMinFlop)) return p;
    // The smallest tile with all tiles on the chip at once, one a CU (two or four
    // groups of waves share its K: alone a group waits for its loads); past that
    // 128 x 128, two a CU.  us in 64 x 64, 64 x 128, 128 x 128 by two groups, 128 x
    // 128: TN 784 x 1024 x 8192 142, 231, 285, 413 (fp32 167); 1999 x 777 x 1531 69,
    // 46, 65, 82 (104); TN 1003 x 2050 x 3000 163, 180, 114, 157 (267); 3000 x 2050 x
    // 1003 164, 130, 99, 92 (211).  256 x 128 and 256 x 256 (spilling) gave NT 8192 x
    // 4096 x 4096 1356 and 1345 against 1435 in 128 x 128, and less of everything else.
    const size_t cus = static_cast<size_t>(device_cu_count());
    auto fits = [&](size_t bm, size_t bn, int groups) {
        if (M < bm || N < bn) return false;
        const size_t tiles = (M + bm - 1) / bm * ((N + bn - 1) / bn) * batches;
        if (groups > 1 ? tiles > cus : tiles > lim) return false;
        p.on = static_cast<double>(M) * N * batches >= 0.45 * bm * bn * tiles;  // (the rest is computed twice)
        p.bm = static_cast<int>(bm);
        p.bn = static_cast<int>(bn);
        p.groups = groups;
        return true;
    };
    if (!fits(64, 64, 4) && !fits(64, 128, 2) && !fits(128, 128, 2)) fits(128, 128, 1);
    return p;
}

template <bool TA, bool TB, int BM, int BN, int WM, int WN, int KG, int NH>
static void launch_tiles(const GemmArgs &g, int products, hipStream_t s) {
    const bool xf = g.xa.n || g.xb.n, epi = g.bias || g.mask || g.relu;
    dim3 grid(static_cast<unsigned>(products)), block(64 * WM * WN * KG);
    if constexpr (TA && !TB) {
        if (g.colsum) {
            grid.x += static_cast<unsigned>((g.N + kStripCols - 1) / kStripCols);
            if (xf) launch((gemm_split<TA, TB, BM, BN, WM, WN, KG, NH, kEpiNone, true, true>), grid, block, 0, s, g, products);
            else launch((gemm_split<TA, TB, BM, BN, WM, WN, KG, NH, kEpiNone, true, false>), grid, block, 0, s, g, products);
            return;
        }
    }
    if (xf) launch((gemm_split<TA, TB, BM, BN, WM, WN, KG, NH, kEpiAll, false, true>), grid, block, 0, s, g, products);
    else if (epi) launch((gemm_split<TA, TB, BM, BN, WM, WN, KG, NH, kEpiAll, false, false>), grid, block, 0, s, g, products);
    else launch((gemm_split<TA, TB, BM, BN, WM, WN, KG, NH, kEpiNone, false, false>), grid, block, 0, s, g, products);
}

template <bool TA, bool TB>
static void launch_layout(const SplitPlan &plan, const GemmArgs &g, int products, hipStream_t s) {
    if (plan.bm == 128 && plan.groups == 1) launch_tiles<TA, TB, 128, 128, 2, 2, 1, 2>(g, products, s);
    else if (plan.bm == 128) launch_tiles<TA, TB, 128, 128, 2, 2, 2, 2>(g, products, s);
    else if (plan.bn == 128) launch_tiles<TA, TB, 64, 128, 2, 2, 2, 4>(g, products, s);
    else launch_tiles<TA, TB, 64, 64, 2, 2, 4, 1>(g, products, s);
}

int launch_split(const SplitPlan &plan, int ta, int tb, GemmArgs g, unsigned batches, hipStream_t s) {
    g.tiles_m = (g.M + plan.bm - 1) / plan.bm;
    g.tiles_n = (g.N + plan.bn - 1) / plan.bn;
    g.tiles = g.tiles_m * g.tiles_n;
    const int products = g.tiles * static_cast<int>(batches);
    if (!ta && !tb) launch_layout<false, false>(plan, g, products, s);
    else if (!ta) launch_layout<false, true>(plan, g, products, s);
    else if (!tb) launch_layout<true, false>(plan, g, products, s);
    else launch_layout<true, true>(plan, g, products, s);
    return launch_status();
}

}  // namespace tship
