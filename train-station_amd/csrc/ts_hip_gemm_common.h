// What the product kernels share (ts_hip_gemm.hip, ts_hip_gemm_split.hip): the
// argument block, operand transforms, tile order and column-sum strips.
#pragma once

#include "ts_hip_internal.h"

namespace tship {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 16;
constexpr int kGroupM = 8;
constexpr int kXcds = 8;

// Column swizzle of LDS row k: bit 4 from the k-quad, bit 5 from k's parity.
__device__ __forceinline__ int swz(int k) { return (((k >> 2) & 3) << 4) ^ ((k & 1) << 5); }

constexpr int kMaxBatchRank = 6;

// An elementwise transform of one operand, applied to each element as it is
// loaded (ts_hip_operand_xf; n == 0: none).  It maps +0 to +0, so the zeros
// that pad a partial k tile stay zeros.
struct OperandXf {
    int n;
    uint8_t code[TS_HIP_XF_MAX_OPS];
    float imm[TS_HIP_XF_MAX_OPS];
};

// A transform read once into scalar registers (the op codes packed in one
// word), so applying it reads no memory.
struct XfRegs {
    int n;
    uint32_t codes;
    float c0, c1, c2, c3;
};
__device__ __forceinline__ XfRegs xf_load(const OperandXf &x) {
    XfRegs r;
    r.n = x.n;
    r.codes = static_cast<uint32_t>(x.code[0]) | (static_cast<uint32_t>(x.code[1]) << 8) |
              (static_cast<uint32_t>(x.code[2]) << 16) | (static_cast<uint32_t>(x.code[3]) << 24);
    r.c0 = x.imm[0];
    r.c1 = x.imm[1];
    r.c2 = x.imm[2];
    r.c3 = x.imm[3];
    return r;
}

// The ops of the transform in order on every element (at(e), E of them),
// each one fp32 operation as the elementwise kernel of the same op computes
// it.  The op's case is chosen once per op (a uniform branch) with the
// elements looped inside it: a switch per element multiplied the kernels'
// code (and compile time) by the element count.
#define TS_XF_EACH(expr) \
    _Pragma("unroll") for (int e = 0; e < E; ++e) { float &x = at(e); x = (expr); } break
template <int E, class At>
__device__ __forceinline__ void xf_each(const XfRegs &xf, At &&at) {
    for (int i = 0; i < xf.n; ++i) {  // uniform
        const uint32_t code = (xf.codes >> (8 * i)) & 255u;
        const float c = i == 0 ? xf.c0 : i == 1 ? xf.c1 : i == 2 ? xf.c2 : xf.c3;
        switch (code) {
            case TS_HIP_XF_ADD_S: TS_XF_EACH(x + c);
            case TS_HIP_XF_SUB_S: TS_XF_EACH(x - c);
            case TS_HIP_XF_MUL_S: TS_XF_EACH(x * c);
            case TS_HIP_XF_DIV_S: TS_XF_EACH(x / c);
            case TS_HIP_XF_RSUB_S: TS_XF_EACH(c - x);
            case TS_HIP_XF_RDIV_S: TS_XF_EACH(c / x);
            case TS_HIP_XF_RELU: TS_XF_EACH(x > 0.0f ? x : 0.0f);
            case TS_HIP_XF_RELU_BWD_S: TS_XF_EACH(x > 0.0f ? c : 0.0f);
            default: TS_XF_EACH(x * x);  // TS_HIP_XF_SQUARE
        }
    }
}
#undef TS_XF_EACH

template <int N>
__device__ __forceinline__ void xf_array(const XfRegs &xf, float (&v)[N]) {
    if (xf.n) xf_each<N>(xf, [&](int e) -> float & { return v[e]; });
}

template <int NF>
__device__ __forceinline__ void xf_regs(const XfRegs &xf, f4v_t (&reg)[NF]) {
    if (!xf.n) return;  // uniform
    float v[4 * NF];
#pragma unroll
    for (int e = 0; e < 4 * NF; ++e) v[e] = reg[e / 4][e % 4];
    xf_each<4 * NF>(xf, [&](int e) -> float & { return v[e]; });
#pragma unroll
    for (int e = 0; e < 4 * NF; ++e) reg[e / 4][e % 4] = v[e];
}

struct GemmArgs {
    const float *A;
    const float *B;
    float *C;
    int M, N, K, lda, ldb, ldc;
    int tiles_m, tiles_n;
    int vec;  // both operands 16-byte aligned with leading dimensions % 4 == 0
    // Batched form (batch_rank > 0): workgroup b computes tile b % tiles of
    // batch b / tiles; a batch's coordinates (row-major over bdims) select
    // A + sum(c_k * sa[k]) and B + sum(c_k * sb[k]) (0 strides on broadcast
    // axes), and C + batch * sc.
    int batch_rank;
    int tiles;  // tiles_m * tiles_n
    int bdims[kMaxBatchRank];
    long long sa[kMaxBatchRank], sb[kMaxBatchRank];
    long long sc;
    // Epilogue (plain form only; all null / 0 for a bare product): the stored
    // value is the product, plus bias[j] when bias is set, then v > 0 ? v : +0 as
    // relu does when relu is set, then kept only where mask[i*ldc + j] > 0
    // (relu's backward with its saved output) when mask is set.
    const float *bias;
    const float *mask;
    int relu;
    // Column sums of B (trans_b == 0; the bias gradient beside a weight
    // gradient) in the column sum's fixed order.  The LDS-DMA kernel writes
    // the sum of each chunk of kColsumRows rows to colsum_part[chunk][n] (f64)
    // from the B tiles it stages anyway -- chunk c by the workgroups of tile
    // row c % tiles_m, so the work is spread over the grid -- and a pass after
    // the product adds the chunks into colsum[n]; the register-staged tiles
    // append a workgroup per 16 columns to their grid, the narrow kernel's
    // first workgroup and the skinny kernel's slice sum add B's columns as
    // they go.  Null: none.
    float *colsum;
    double *colsum_part;
    int kslice;  // skinny products: k rows per slice
    // operand transforms (register-staged tiles, the narrow and one-k-tile
    // kernels and the column strips apply them; the others take none)
    OperandXf xa, xb;
    // The sum (mean: / (float)sum_n) of the sum_n floats at sum_x, each put
    // through sum_xf first, into sum_out[0] with the bits of ts_hip_sum over
    // the transformed values: one workgroup appended to the grid of a product
    // with column sums (after the register-staged tiles' strips, or as the
    // narrow kernel's last row block) runs sum_in_workgroup over sum_blocks
    // first-pass workgroups.  Null sum_out: none.
    const float *sum_x;
    float *sum_out;
    size_t sum_n;
    int sum_mean, sum_blocks;
    OperandXf sum_xf;
    // Epilogue subtraction (narrow kernel only): after the bias, v = v -
    // sub[i*ldc + j] (laid out as C).  Null: none.
    const float *sub;
};

// The epilogue kinds of a product's kernels; kEpiBiasRelu ignores the mask, so
// a kernel that never sees one keeps no registers for it.
enum : int { kEpiNone = 0, kEpiBiasRelu = 1, kEpiAll = 2 };

// Store of a wave's FM x FN accumulator blocks, the wave tile's corner at
// (i0, j0).  Accumulator layout of v_mfma_f32_32x32x2_f32: lane l, register
// r holds C[8*(r/4) + 4*(l/32) + r%4][l%32] of the 32x32 block.  With EPI the
// stored value is the product, plus bias[j], then v > 0 ? v : +0 (relu), then
// kept only where mask[i*ldc + j] > 0: the unfused ops in their order.  A row
// of blocks at a time: its mask is loaded before its first store, so those
// loads overlap each other (every block's at once would need a register per
// output element).  EPI is one of the kinds above.
// s_waitcnt immediate for vmcnt(0) with expcnt and lgkmcnt left at their
// maxima (gfx9 encoding: vmcnt[3:0], expcnt[6:4], lgkmcnt[11:8]).
constexpr int kWaitVm0 = 0x0F70;

template <int EPI, int FM, int FN>
__device__ __forceinline__ void store_tile(const GemmArgs &g, const floatx16 (&acc)[FM][FN], float *Cp, int i0,
                                           int j0, int lrow, int lhalf) {
    float bj[FN];  // bias of the lane's column in each block column
#pragma unroll
    for (int b = 0; b < FN; ++b) {
        const int j = j0 + b * 32 + lrow;
        bj[b] = (EPI != kEpiNone && g.bias && j < g.N) ? g.bias[j] : 0.0f;
    }
    // Wait for the bias here, once.  Left to the compiler, the wait lands in
    // every guarded store's branch, and as a full vmcnt(0) (the load may be
    // pending on the path that skipped the previous store), so each store
    // would wait for all earlier ones to complete.
    if (EPI != kEpiNone) __builtin_amdgcn_s_waitcnt(kWaitVm0);
    auto value = [&](float v, int b, float m) {
        if (EPI != kEpiNone) {
            if (g.bias) v = v + bj[b];
            if (g.relu) v = v > 0.0f ? v : 0.0f;
            if (EPI == kEpiAll && g.mask) v = m > 0.0f ? v : 0.0f;
        }
        return v;
    };
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        float mk[FN][16];
        if (EPI == kEpiAll && g.mask) {
#pragma unroll
            for (int b = 0; b < FN; ++b) {
                const int j = j0 + b * 32 + lrow;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int i = i0 + a * 32 + 8 * (r >> 2) + 4 * lhalf + (r & 3);
                    mk[b][r] = (i < g.M && j < g.N) ? g.mask[(size_t)i * g.ldc + j] : 0.0f;
                }
            }
            __builtin_amdgcn_s_waitcnt(kWaitVm0);  // as for the bias
        }
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            const int j = j0 + b * 32 + lrow;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = i0 + a * 32 + 8 * (r >> 2) + 4 * lhalf + (r & 3);
                if (i < g.M && j < g.N) Cp[(size_t)i * g.ldc + j] = value(acc[a][b][r], b, mk[b][r]);
            }
        }
        if (EPI == kEpiAll) __builtin_amdgcn_sched_barrier(0);
    }
}

// Staging of one operand tile: logical [BK][R] (k-major), R = 64, 128 or 256
// rows of the operand's non-k index.  KCONTIG: k is the contiguous index in
// memory (row-major A, or B^T); otherwise the R index is contiguous.
template <int R, int NT, bool KCONTIG>
struct Stage {
    static constexpr int NF = R * kBK / 4 / NT;  // float4 per thread
    static_assert(NF >= 1 && R % 16 == 0, "tile does not divide over the workgroup");

    // float4 number f -> (row, first k) of that float4 in the tile
    static __device__ __forceinline__ void coords(int f, int &row, int &kk) {
        if (KCONTIG) {
            // a wave instruction covers 16 rows x 4 k-quads: 16 lanes per k-quad
            const int grp = f >> 6, l = f & 63;
            const int rb = grp % (R / 16), kb = grp / (R / 16);
            row = rb * 16 + (l & 15);
            kk = 4 * (kb * 4 + (l >> 4));
        } else {
            kk = f / (R / 4);
            row = 4 * (f % (R / 4));
        }
    }

    // a tile with every k inside: one dwordx4 per float4, the row index kept
    // inside the operand (rows past an M / N edge feed outputs that are never
    // stored, so any in-bounds values serve).  Needs the
    // layout of g.vec (16-byte aligned, ld % 4 == 0): for a k-contiguous
    // operand a row is clamped to rows - 1; otherwise a float4 of 4 rows
    // starts at most at (rows - 1) & ~3, which ld >= rows rounded up to 4
    // keeps inside the row.
    static __device__ __forceinline__ void load_clamped(const float *__restrict__ P, int ld, int rows, int r0,
                                                        int k0, f4v_t (&reg)[NF]) {
#pragma unroll
        for (int s = 0; s < NF; ++s) {
            int row, kk;
            coords(s * NT + static_cast<int>(threadIdx.x), row, kk);
            if (KCONTIG) {
                const int r = min(r0 + row, rows - 1);
                reg[s] = *reinterpret_cast<const f4v_t *>(P + (size_t)r * ld + (k0 + kk));
            } else {
                const int r = min(r0 + row, (rows - 1) & ~3);
                reg[s] = *reinterpret_cast<const f4v_t *>(P + (size_t)(k0 + kk) * ld + r);
            }
        }
    }

    // edge tile: element loads with bounds checks, zeros outside
    static __device__ __forceinline__ void load_guarded(const float *__restrict__ P, int ld, int rows,
                                                        int K, int r0, int k0, f4v_t (&reg)[NF]) {
#pragma unroll
        for (int s = 0; s < NF; ++s) {
            int row, kk;
            coords(s * NT + static_cast<int>(threadIdx.x), row, kk);
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int gr = KCONTIG ? r0 + row : r0 + row + c;
                const int gk = KCONTIG ? k0 + kk + c : k0 + kk;
                v[c] = (gr < rows && gk < K)
                           ? (KCONTIG ? P[(size_t)gr * ld + gk] : P[(size_t)gk * ld + gr])
                           : 0.0f;
            }
            reg[s] = f4v_t{v[0], v[1], v[2], v[3]};
        }
    }

    static __device__ __forceinline__ void store(float *S, const f4v_t (&reg)[NF]) {
#pragma unroll
        for (int s = 0; s < NF; ++s) {
            int row, kk;
            coords(s * NT + static_cast<int>(threadIdx.x), row, kk);
            if (KCONTIG) {
#pragma unroll
                for (int c = 0; c < 4; ++c) S[(kk + c) * R + (row ^ swz(kk + c))] = reg[s][c];
            } else {
                *reinterpret_cast<f4v_t *>(&S[kk * R + (row ^ swz(kk))]) = reg[s];
            }
        }
    }
};

// The operand offsets of a batch (GemmArgs::batch_rank > 0).  The loop is
// unrolled with constant indices so the argument arrays stay in SGPRs.
__device__ __forceinline__ void batch_offsets(const GemmArgs &g, int batch, long long &oa, long long &ob) {
    oa = ob = 0;
#pragma unroll
    for (int k = kMaxBatchRank - 1; k >= 0; --k) {
        if (k < g.batch_rank) {
            const int c = batch % g.bdims[k];
            batch /= g.bdims[k];
            oa += c * g.sa[k];
            ob += c * g.sb[k];
        }
    }
}

// Tile coordinates of workgroup b of a G-tile grid (see the file comment).
__device__ inline void tile_coords(int tiles_m, int tiles_n, int b, int &tm, int &tn) {
    const int G = tiles_m * tiles_n;
    const int xcd = b % kXcds;
    int prefix = 0;
    for (int y = 0; y < xcd; ++y) prefix += (G - y + kXcds - 1) / kXcds;
    const int logical = prefix + b / kXcds;
    const int group_size = kGroupM * tiles_n;
    const int group = logical / group_size;
    const int first_m = group * kGroupM;
    int gsz = tiles_m - first_m;
    if (gsz > kGroupM) gsz = kGroupM;
    const int in_group = logical - group * group_size;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

// Column sums of B ([K][N], trans_b == 0) for 16 columns, j0 .. j0+15, in
// the column sum's order, by one workgroup of NT threads: in rounds of
// NT/16 chunks, thread (chunk q, column j) adds its chunk's rows from +0 in
// f64 (16 rows in flight at a time, rows past K read in bounds and not
// added), then thread j adds the round's groups of chunk sums, each from +0,
// into its running total, and finally stores it.
constexpr int kStripCols = 16;

template <int NT, bool XF>
__device__ __forceinline__ void colsum_strip(const GemmArgs &g, int j0) {
    constexpr int R = static_cast<int>(kColsumRows), G = static_cast<int>(kColsumGroup), RC = NT / kStripCols;
    static_assert(RC * kStripCols == NT && RC % G == 0, "a round holds whole groups of chunks");
    __shared__ double cs[RC][kStripCols];
    const int t = static_cast<int>(threadIdx.x), q = t / kStripCols, j = t % kStripCols;
    const int col = min(j0 + j, g.N - 1);
    const int chunks = (g.K + R - 1) / R;
    const XfRegs xfb = xf_load(g.xb);
    double total = 0.0;
    for (int c0 = 0; c0 < chunks; c0 += RC) {  // uniform
        const int r0 = (c0 + q) * R;
        double sum = 0.0;
        for (int rb = 0; rb < R; rb += 16) {
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = g.B[(size_t)min(r0 + rb + r, g.K - 1) * g.ldb + col];
            if constexpr (XF) xf_array(xfb, v);  // the rows past K are transformed too, and not added
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (r0 + rb + r < g.K) sum += (double)v[r];
        }
        cs[q][j] = sum;
        __syncthreads();
        if (t < kStripCols) {
#pragma unroll
            for (int h = 0; h < RC / G; ++h) {
                double grp = 0.0;
#pragma unroll
                for (int i = 0; i < G; ++i) grp += cs[h * G + i][t];
                total += grp;
            }
        }
        __syncthreads();
    }
    if (t < kStripCols && j0 + t < g.N) g.colsum[j0 + t] = static_cast<float>(total);
}

// One BM x BN tile at (i0, j0) of a product on the fp32 matrix instructions,
// by a workgroup of WM x WN waves: the loop over K, then the store with its
// epilogue.  EPI: the epilogue kind applied at the store
// (a separate instantiation per kind, so the bare product keeps its register
// allocation).  PF: operand tiles prefetched into registers ahead of the LDS
// stage (deeper for small tiles, whose k-steps are too short to cover a global
// load).  VEC (operands 16-byte aligned, leading dimensions % 4 == 0): the loop
// runs the whole k tiles with dwordx4 loads whose rows are clamped into the
// operand (rows past an M / N edge feed outputs that are never stored), and a
// partial last tile follows it with element loads; otherwise every tile takes
// bounds-checked element loads (zeros outside).  LDS: As 2 * kBK * BM floats,
// Bs 2 * kBK * BN.
template <bool TA, bool TB, int BM, int BN, int WM, int WN, int EPI, int PF, bool VEC, bool XF>
__device__ __forceinline__ void fp32_tile(const GemmArgs &g, const float *Ap, const float *Bp, float *Cp, int K, int i0,
                                          int j0, float (*As)[kBK * BM], float (*Bs)[kBK * BN]) {
    constexpr int NT = 64 * WM * WN;
    constexpr int TMW = BM / WM, TNW = BN / WN;  // wave tile
    constexpr int FM = TMW / 32, FN = TNW / 32;  // 32x32 accumulators per wave
    using SA = Stage<BM, NT, !TA>;                // A is k-contiguous unless transposed
    using SB = Stage<BN, NT, TB>;                 // B is k-contiguous only when transposed
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int lrow = lane & 31, lhalf = lane >> 5;
    const XfRegs xfa = XF ? xf_load(g.xa) : XfRegs{}, xfb = XF ? xf_load(g.xb) : XfRegs{};

    floatx16 acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    // One k tile from LDS: every operand read, then the MFMAs in k order
    // (the reads complete in order, so each MFMA waits only for its own).
    auto mma = [&](const float *Ac, const float *Bc) {
        float af[kBK / 2][FM], bf[kBK / 2][FN];
#pragma unroll
        for (int s = 0; s < kBK / 2; ++s) {
            const int k = 2 * s + lhalf;
#pragma unroll
            for (int a = 0; a < FM; ++a) af[s][a] = Ac[k * BM + ((wm * TMW + a * 32 + lrow) ^ swz(k))];
#pragma unroll
            for (int b = 0; b < FN; ++b) bf[s][b] = Bc[k * BN + ((wn * TNW + b * 32 + lrow) ^ swz(k))];
        }
#pragma unroll
        for (int s = 0; s < kBK / 2; ++s)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[s][a], bf[s][b], acc[a][b], 0, 0, 0);
    };

    // Every step issues the same loads (steps past the end re-load the last
    // tile), so the compiler's load counters stay exact and the PF-deep
    // register ring really has PF tiles of loads in flight.
    const int nt = VEC ? K / kBK : (K + kBK - 1) / kBK;  // tiles of the loop
    f4v_t ra[PF][SA::NF], rb[PF][SB::NF];
    auto load = [&](int t, f4v_t(&a)[SA::NF], f4v_t(&b)[SB::NF]) {
        const int k0 = min(t, nt - 1) * kBK;
        if (VEC) {
            SA::load_clamped(Ap, g.lda, g.M, i0, k0, a);
            SB::load_clamped(Bp, g.ldb, g.N, j0, k0, b);
        } else {
            SA::load_guarded(Ap, g.lda, g.M, K, i0, k0, a);
            SB::load_guarded(Bp, g.ldb, g.N, K, j0, k0, b);
        }
    };

    if (nt > 0) {
        load(0, ra[0], rb[0]);
        if constexpr (XF) {
            xf_regs(xfa, ra[0]);
            xf_regs(xfb, rb[0]);
        }
        SA::store(As[0], ra[0]);
        SB::store(Bs[0], rb[0]);
#pragma unroll
        for (int p = 0; p < PF; ++p) load(1 + p, ra[p], rb[p]);
        __syncthreads();

        for (int kt0 = 0; kt0 < nt; kt0 += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int kt = kt0 + u;
                if (kt >= nt) break;  // uniform
                const int cur = kt & 1;
                // LDS[cur] holds tile kt: its operands are read and its MFMAs
                // issued; slot u (tile kt+1, past the end a re-load) goes to
                // buffer cur^1, last read before the previous barrier, and
                // slot u then takes tile kt+1+PF.  One basic block, so the
                // scheduler can place the stores and loads in the MFMAs'
                // shadow (a wave issues in order).
                mma(As[cur], Bs[cur]);
                if constexpr (XF) {
                    xf_regs(xfa, ra[u]);
                    xf_regs(xfb, rb[u]);
                }
                SA::store(As[cur ^ 1], ra[u]);
                SB::store(Bs[cur ^ 1], rb[u]);
                load(kt + 1 + PF, ra[u], rb[u]);
                __syncthreads();
            }
        }
    }
    if (VEC && nt * kBK < K) {  // the partial last k tile (uniform)
        f4v_t pa[SA::NF], pb[SB::NF];
        SA::load_guarded(Ap, g.lda, g.M, K, i0, nt * kBK, pa);
        SB::load_guarded(Bp, g.ldb, g.N, K, j0, nt * kBK, pb);
        if constexpr (XF) {
            xf_regs(xfa, pa);
            xf_regs(xfb, pb);
        }
        SA::store(As[0], pa);
        SB::store(Bs[0], pb);
        __syncthreads();
        mma(As[0], Bs[0]);
    }
    store_tile<EPI, FM, FN>(g, acc, Cp, i0 + wm * TMW, j0 + wn * TNW, lrow, lhalf);
}

// Register prefetch depth per tile size: one tile ahead for 256x256 tiles
// (a k-step of 8 waves' 128x64 blocks is long), four for the smaller ones.
template <int BM>
constexpr int prefetch_tiles() { return BM >= 256 ? 1 : 4; }

// ---- products on the bf16 matrix cores (ts_hip_gemm_split.hip) --------------------

// Whether a product takes them (every entry point asks here), its tile (bm x bn
// of C per workgroup) and the groups of waves that share a tile's K.
struct SplitPlan {
    bool on = false;
    int bm = 0, bn = 0, groups = 1;
};
SplitPlan split_plan(int trans_a, int trans_b, size_t M, size_t N, size_t K, size_t batches);
// The product; g as for the fp32 kernels (no sum_out).
int launch_split(const SplitPlan &plan, int ta, int tb, GemmArgs g, unsigned batches, hipStream_t s);

}  // namespace tship
