// Choice and launch of the products on the f16 matrix cores (the kernels and
// their reasons: ts_hip_gemm_split.h).
#include "ts_hip_gemm_split.h"

#include <algorithm>

namespace tship {

// Products of fewer operations than this stay on the fp32 instructions.  Against
// the fp32 kernels (us, theirs and these): 1024 x 1024 x 784, 1.6e9: 21, 28; 1024 x
// 1024 x 1024, 2.1e9: 26, 29; 2000 x 300 x 2000, 2.4e9: 44, 39; 640 x 640 x 3000,
// 2.5e9: 64, 32.  Where a size is no multiple of four those load element by
// element: 1000 x 1000 x 500, 1.0e9, aligned: 15, 27; 999 x 777 x 1001, 1.6e9: 39,
// 33; 1500 x 700 x 900: 36, 31.
constexpr double kSplitMinFlop = 2.2e9, kSplitMinFlopRagged = 1.5e9;
// Floats of partial products at most (they stay in the caches).
constexpr size_t kSplitMaxPartial = size_t(1) << 23;
constexpr size_t kSplitMaxScan = size_t(1) << 20;  // floats of a scan at most

// The scan of one operand's slice: chunks of k, k per chunk and workgroups.
static void scan_grid(bool kcontig, size_t rows, size_t K, size_t slices, int &chunks, int &kc, int &blocks) {
    if (kcontig) {
        chunks = 1;
        kc = static_cast<int>(K);
        blocks = static_cast<int>((rows + kScanRows - 1) / kScanRows);
        return;
    }
    const size_t cols = (rows + kScanCols - 1) / kScanCols;
    const size_t c = std::max<size_t>(1, std::min({1024 / (cols * slices), size_t(kScanChunks), (K + 63) / 64}));
    kc = static_cast<int>((K + c - 1) / c);
    chunks = static_cast<int>((K + kc - 1) / kc);
    blocks = static_cast<int>(cols) * chunks;
}

SplitPlan split_plan(size_t M, size_t N, size_t K, size_t batches) {
    SplitPlan p;
    const size_t lim = size_t(1) << 23;  // exponent sums and lane offsets in 32 bits
    if (M < 64 || N < 64 || K < 64 || M > lim || N > lim || K > lim || K * N <= 16384 || batches == 0) return p;
    const bool ragged = M % 4 != 0 || N % 4 != 0 || K % 4 != 0;
    if (2.0 * M * N * K * batches < (ragged ? kSplitMinFlopRagged : kSplitMinFlop)) return p;
    auto tiles = [&](size_t t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
    const size_t cus = static_cast<size_t>(device_cu_count());
    const size_t t256 = tiles(256), t128 = tiles(128);
    if (M * N < t128 * 7400) return p;  // less than 45% of 128 x 128 tiles used
    // 256 x 256 tiles once they fill the chip (2048 x 4096 x 1024, half the chip:
    // 80 us against 60 in 128 x 128, before the scan), unless their padding is
    // more than a tenth over that of 128 x 128
    p.tile = t256 * batches >= cus && 40 * t256 <= 11 * t128 ? 256 : 128;
    const size_t nt = p.tile == 256 ? t256 : t128;
    if (nt * batches > 0x7fffffffULL / 16) return p;
    p.on = true;
    if (p.tile == 128 && batches == 1 && nt < cus) {
        // fewer tiles than CUs: two workgroups a CU, slices of at least 256 k (a
        // lone workgroup is bound by its latencies: 1531 x 777 x 1999 whole took
        // 81 us, in slices 50 with their sum)
        const size_t ldp = (N + 3) & ~size_t(3);
        size_t sl = std::min({2 * cus / nt, size_t(kSplitMaxSlices), K / 256, kSplitMaxPartial / (M * ldp)});
        for (; sl > 1; --sl) {
            const size_t ks = ((K + sl - 1) / sl + kSplitK - 1) / kSplitK * kSplitK;
            if (ks >= K || (K - 1) % ks + 1 < kSplitK) continue;  // the last slice holds a whole stage too
            p.slices = static_cast<int>((K + ks - 1) / ks);
            p.kslice = static_cast<int>(ks);
            p.partial_floats = p.slices * M * ldp;
            break;
        }
    }
    if (batches == 1) {
        int cm, cn, unused;
        const size_t slices = static_cast<size_t>(p.slices), ks = p.kslice ? static_cast<size_t>(p.kslice) : K;
        scan_grid(false, M, ks, slices, cm, unused, unused);  // the layout that takes more
        scan_grid(false, N, ks, slices, cn, unused, unused);
        p.scan_floats = sizeof(SplitRow) / sizeof(float) * slices * (cm * M + cn * N);
        if (p.scan_floats > kSplitMaxScan) p.scan_floats = 0;
    }
    return p;
}

template <bool TA, bool TB>
static void launch_layout(const SplitPlan &plan, const GemmArgs &g, int products, const SplitScanArgs &scans,
                          hipStream_t s) {
    const bool xf = g.xa.n || g.xb.n, epi = g.bias || g.mask || g.relu;
    if (scans.a) {
        const dim3 sg(static_cast<unsigned>(scans.blocks_a + scans.blocks_b) * static_cast<unsigned>(plan.slices));
        if (xf) launch((split_scan<TA, TB, true>), sg, dim3(256), 0, s, g, scans);
        else launch((split_scan<TA, TB, false>), sg, dim3(256), 0, s, g, scans);
    }
    dim3 grid(static_cast<unsigned>(products));
    if (plan.tile == 256) {
        if (epi) launch((gemm_split<TA, TB, 256, 256, 2, 4, 1, kEpiAll, false, false>), grid, dim3(512), 0, s, g, products, scans);
        else launch((gemm_split<TA, TB, 256, 256, 2, 4, 1, kEpiNone, false, false>), grid, dim3(512), 0, s, g, products, scans);
        return;
    }
    if constexpr (TA && !TB) {
        if (g.colsum) {
            grid.x += static_cast<unsigned>((g.N + kStripCols - 1) / kStripCols);
            if (xf) launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiNone, true, true>), grid, dim3(256), 0, s, g, products, scans);
            else launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiNone, true, false>), grid, dim3(256), 0, s, g, products, scans);
            return;
        }
    }
    if (xf && epi) launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiAll, false, true>), grid, dim3(256), 0, s, g, products, scans);
    else if (xf) launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiNone, false, true>), grid, dim3(256), 0, s, g, products, scans);
    else if (epi) launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiAll, false, false>), grid, dim3(256), 0, s, g, products, scans);
    else launch((gemm_split<TA, TB, 128, 128, 2, 2, 2, kEpiNone, false, false>), grid, dim3(256), 0, s, g, products, scans);
}

int launch_split(const SplitPlan &plan, int ta, int tb, GemmArgs g, unsigned batches, float *partial, float *scan,
                 hipStream_t s) {
    g.tiles_m = (g.M + plan.tile - 1) / plan.tile;
    g.tiles_n = (g.N + plan.tile - 1) / plan.tile;
    g.tiles = g.tiles_m * g.tiles_n;
    g.kslice = plan.kslice;
    const int products = g.tiles * plan.slices * static_cast<int>(batches);
    const GemmArgs whole = g;
    if (plan.slices > 1) {  // bare, one after another
        g.C = partial;
        g.ldc = (g.N + 3) & ~3;
        g.bias = g.mask = nullptr;
        g.relu = 0;
    }
    SplitScanArgs p{};
    if (scan) {
        const size_t ks = plan.kslice ? static_cast<size_t>(plan.kslice) : static_cast<size_t>(g.K);
        const size_t slices = static_cast<size_t>(plan.slices);
        scan_grid(!ta, static_cast<size_t>(g.M), ks, slices, p.chunks_a, p.kc_a, p.blocks_a);
        scan_grid(tb, static_cast<size_t>(g.N), ks, slices, p.chunks_b, p.kc_b, p.blocks_b);
        p.a = reinterpret_cast<SplitRow *>(scan);
        p.b = p.a + slices * p.chunks_a * g.M;
    }
    if (!ta && !tb) launch_layout<false, false>(plan, g, products, p, s);
    else if (!ta) launch_layout<false, true>(plan, g, products, p, s);
    else if (!tb) launch_layout<true, false>(plan, g, products, p, s);
    else launch_layout<true, true>(plan, g, products, p, s);
    if (plan.slices > 1)
        launch(split_sum, dim3(static_cast<unsigned>((g.N + 255) / 256), static_cast<unsigned>((g.M + 3) / 4)), dim3(256),
               0, s, static_cast<const float *>(partial), plan.slices, g.ldc, whole);
    return launch_status();
}

}  // namespace tship
