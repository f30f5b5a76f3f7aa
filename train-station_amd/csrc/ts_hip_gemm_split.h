// fp32 products on the f16 matrix cores (the kernels; ts_hip_gemm_split.hip
// chooses and launches them).
//
// The fp32 matrix instructions bound the large products at 157 TFLOP/s; the
// f16 ones run 16 times as fast.  An fp32 value scaled into f16's range is the
// sum of two f16 values to within 2^-24 of itself, h = f16(v) (11 bits) and
// l = f16(v - h) (the next 11, and the sign of the remainder), so
//   a b = ha hb + ha lb + la hb   (la lb < 2^-24 |a b| left out),
// three f16 products whose exact sums of 32 are added in fp32.  The error per
// term is that of rounding its factors once more, and the running sum is
// rounded 3/32 times per term instead of once, so the result is closer to the
// exact one than the fp32 instructions' (measured below).
//
// Range.  Each row of op(A) and column of op(B) of a tile is scaled by the power
// of two that puts its largest magnitude into [2^14, 2^15); the scales'
// exponents are taken back from the finished sums (ldexp, one rounding).  An
// element's error is then at most 2^-24 of itself or 2^-40 of its row's
// largest, whichever is larger.  A workgroup first scans its rows and columns
// over its k for the largest magnitude and the mean exponent of the non-zero
// elements (a fifth to a quarter of the kernel's time: it reads what the product
// will, from L2).  A tile with a row or column that holds an
// infinity, that is too small to scale, or whose mean lies more than
// kSplitSpread binades below its largest (2^-40 of the largest would be more
// than 2^-25 of an ordinary element) runs on the fp32 instructions instead
// (fp32_tile).  Where the caller gave a workspace the scan is a launch of its own.
// A NaN needs no care: it is NaN in h, and so in the sums it enters.
//
// Sign.  The f16 instruction drops the low bits of its sum downwards: over a
// long k the results lie about 1e-7 of their typical size too low (K = 4096),
// less than the rounding of either kind but the same way in every element and
// call.  So the last 3/8 of the stages add up the negated product to the
// negated sum: their error points the other way, and with the running sum
// growing as sqrt(k) the two parts' cancel (3/8: 1 - 2^(-2/3)).
//
// Tiles.  BM x BN per workgroup in k stages of 32, two LDS stages.  Global
// loads of stage t + 2 go to registers while stage t + 1's registers are
// scaled, split and written to LDS and stage t's fragments feed the matrix
// cores; one barrier per stage, before the stage's last block of rows so that
// its MFMAs cover the first reads of the next stage.
//
// Measured (us; fp32 instructions before, scanning in the workgroups, with a scan
// of its own): NT 8192 x 4096 x 4096 1896, 900, 740 (372 TFLOP/s; the matrix cores
// busy 63% of the cycles at the 1.7 GHz they reach); TN 4096 x 4096 x 8192 1892,
// 865, 739; NN 2048 x 4096 x 1024 149, 85, 71; TN 1003 x 2050 x 3000 267, 94, 80; NT
// 1999 x 1531 x 777 104, 54, 49; 64 x NN 1024 x 128 x 1024 (no workspace) 268, 158.  Error against 64 bits, of normal data: K = 4096 1.14e-6,
// 7.1e-7; K = 1024 5.7e-7, 3.6e-7.
//
// LDS.  An operand stage is h then l, each [row block of 16][64 chunks of 16
// bytes]: chunk q * 16 + (i ^ X[q]) of a block holds, for its row i, the k 4q ..
// 4q + 3 and 16 + 4q .. 16 + 4q + 3 (the order of k within a stage is free as
// long as both operands share it, and this one lets four lanes read 64
// consecutive bytes of a k-contiguous row).  A fragment (lane (i, q), eight k)
// is one 16-byte read; X = {0, 12, 4, 8} keeps the reads and the writes of a
// k-contiguous operand free of bank conflicts.  B's rows, and a row-contiguous
// A's, are interleaved: block b of a group of G rows holds its rows i * G/16 +
// b, so a lane owns neighbouring columns of C and stores them together, and
// the four rows of a float4 go to four blocks at one address.  (An interleaved
// k-contiguous operand writes those four blocks side by side: there the chunk
// is also XORed with the block's number.)
#pragma once

#include "ts_hip_gemm_common.h"

typedef _Float16 h2v_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4v_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8v_t __attribute__((ext_vector_type(8)));
typedef float f2v_t __attribute__((ext_vector_type(2)));
// four floats at any 4-byte address (gfx950 loads them with one instruction)
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

namespace tship {

template <bool V>
struct BoolTag {
    static constexpr bool value = V;
};

constexpr int kSplitK = 32;
constexpr int kSplitSpread = 15;
constexpr int kScanDepth = 2;  // stages in flight in the scan (1 to 3 measured alike)
constexpr int kSplitTopExp = 127 + 14;  // the scaled exponent field of a row's largest element

// What the scan knows of a tile's rows: the largest magnitude's bits, and the
// exponent fields' sum and count over the non-zero elements (a subnormal counts
// as zero).
template <int R>
struct SplitScan {
    unsigned top[R], sum[R], cnt[R];
};

// ---- staging ----------------------------------------------------------------------

__device__ __forceinline__ int split_x(int q) { return 12 * (q & 1) ^ 4 * ((q >> 1) & 1); }

// two values times their scales, split (a power of two times a value and the
// remainder of its rounding are exact)
__device__ __forceinline__ void split2(float a, float sa, float b, float sb, h2v_t &h, h2v_t &l) {
    const f2v_t v = {a * sa, b * sb};
    h = __builtin_convertvector(v, h2v_t);
    const f2v_t r = {__builtin_fmaf(a, sa, -static_cast<float>(h[0])), __builtin_fmaf(b, sb, -static_cast<float>(h[1]))};
    l = __builtin_convertvector(r, h2v_t);
}

// One operand's staging by NT threads: R rows (groups of G interleaved; G ==
// 16: in order), 32 k.
// KC (k contiguous): a thread's unit is one row and quarter (two float4, one
// 16-byte chunk); else four rows and half a quarter (four float4, a row each
// of k; four 8-byte half chunks).  Rows past the operand repeat its last (their
// outputs are never stored).
template <int R, int G, int NT, bool KC>
struct SplitStage {
    static constexpr int U = KC ? (R * 4 + NT - 1) / NT : (R * 2 + NT - 1) / NT;  // units per thread
    static constexpr int NF = KC ? 2 * U : 4 * U;
    static constexpr int NS = KC ? U : 4 * U;  // scales
    static constexpr int kUnits = KC ? R * 4 : R * 2;
    static_assert(KC ? R * 4 % NT == 0 || NT % (R * 4) == 0 : R * 2 % NT == 0 || NT % (R * 2) == 0, "units");

    static constexpr bool kXor = KC && G > 16;

    // byte address, within a stage's h (or l), of row `row` and k quarter q
    static __device__ __forceinline__ int at(int row, int q) {
        constexpr int F = G / 16;
        const int blk = (row / G) * F + row % F, i = (row % G) / F;
        return blk * 1024 + (q * 16 + (i ^ split_x(q) ^ (kXor ? blk & 3 : 0))) * 16;
    }
    // unit u of thread t; more threads than units: several do the same one
    static __device__ __forceinline__ int unit(int u) { return (u * NT + static_cast<int>(threadIdx.x)) % kUnits; }
    static __device__ __forceinline__ void coords(int u, int &row, int &q, int &half) {
        const int n = unit(u);
        if (KC) {
            row = n >> 2;
            q = n & 3;
            half = 0;
        } else {
            row = 4 * (n % (R / 4));
            q = (n / (R / 4)) >> 1;
            half = (n / (R / 4)) & 1;
        }
    }
    // The row the offsets start from: the tile's first, or where fewer than four
    // are left of the operand its fourth last (not KC), so that no float4 ends
    // past the operand.
    static __device__ __forceinline__ int first(int rows, int r0) { return KC ? r0 : min(r0, rows - 4); }
    // byte offset of a unit's first float4 from row first() and the stage's first k
    static __device__ __forceinline__ void offsets(unsigned (&off)[U], int ld, int rows, int r0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int row, q, half;
            coords(u, row, q, half);
            if (KC) off[u] = static_cast<unsigned>(min(row, rows - 1 - r0)) * static_cast<unsigned>(ld) * 4u + 16u * q;
            else off[u] = static_cast<unsigned>(16 * half + 4 * q) * static_cast<unsigned>(ld) * 4u +
                          4u * static_cast<unsigned>(min(row, rows - 4 - first(rows, r0)));
        }
    }
    // float4 number f of a whole stage
    static __device__ __forceinline__ f4v_t load(const float *base, int ld, const unsigned (&off)[U], int f) {
        const char *p = reinterpret_cast<const char *>(base);
        if (KC) return *reinterpret_cast<const f4u_t *>(p + 64 * (f & 1) + off[f / 2]);
        return *reinterpret_cast<const f4u_t *>(p + (size_t)(f & 3) * ld * 4 + off[f / 4]);
    }
    // the same, any row count and any k: rows clamped one by one, zeros past K
    static __device__ __forceinline__ f4v_t load_edge(const float *P, int ld, int rows, int K, int r0, int k0, int f) {
        int row, q, half;
        coords(KC ? f / 2 : f / 4, row, q, half);
        f4v_t v;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int r = min(r0 + row + (KC ? 0 : c), rows - 1);
            const int k = k0 + 4 * q + (KC ? 16 * (f & 1) + c : 16 * half + (f & 3));
            const int kk = min(k, K - 1);
            const float x = KC ? P[(size_t)r * ld + kk] : P[(size_t)kk * ld + r];
            v[c] = k < K ? x : 0.0f;
        }
        return v;
    }
    // Not KC: the float4 that would end past the operand's last row was loaded
    // from the last four rows: its values moved to their places (the operand
    // has at least four rows).
    static __device__ __forceinline__ void mend(f4v_t (&reg)[NF], int rows, int r0, int u) {
        int row, q, half;
        coords(u, row, q, half);
        const int s = row - min(row, rows - 4 - r0);  // 1..3 for it, 4 and more for those past the operand
#pragma unroll
        for (int f = 4 * u; f < 4 * u + 4; ++f) {
            const f4v_t v = reg[f];
            reg[f][0] = s == 0 ? v[0] : s == 1 ? v[1] : s == 2 ? v[2] : v[3];
            reg[f][1] = s == 0 ? v[1] : s == 1 ? v[2] : v[3];
            reg[f][2] = s == 0 ? v[2] : v[3];
        }
    }
    static __device__ __forceinline__ void scales(float (&sc)[NS], const SplitScan<R> &S) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int row, q, half;
            coords(u, row, q, half);
#pragma unroll
            for (int c = 0; c < NS / U; ++c) sc[u * (NS / U) + c] = __uint_as_float((127u + S.top[row + c]) << 23);
        }
    }
    // A stage's values of unit u into its rows' scan (top's index: scale).
    static __device__ __forceinline__ void scan(const f4v_t (&reg)[NF], int u, float (&top)[NS], unsigned (&sum)[NS],
                                                unsigned (&cnt)[NS]) {
        auto four = [&](float v0, float v1, float v2, float v3, int i) {
            auto e = [](float v) { return __builtin_amdgcn_ubfe(__float_as_uint(v), 23, 8); };
            const unsigned e0 = e(v0), e1 = e(v1), e2 = e(v2), e3 = e(v3);
            top[i] = fmaxf(fmaxf(fmaxf(fmaxf(top[i], fabsf(v0)), fabsf(v1)), fabsf(v2)), fabsf(v3));
            sum[i] = sum[i] + e0 + e1 + (e2 + e3);
            cnt[i] = cnt[i] + min(e0, 1u) + min(e1, 1u) + (min(e2, 1u) + min(e3, 1u));
        };
        if (KC) {
#pragma unroll
            for (int f = 2 * u; f < 2 * u + 2; ++f) four(reg[f][0], reg[f][1], reg[f][2], reg[f][3], u);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                four(reg[4 * u][c], reg[4 * u + 1][c], reg[4 * u + 2][c], reg[4 * u + 3][c], 4 * u + c);
        }
    }
    // the threads' scans of a row joined
    static __device__ __forceinline__ void scan_join(SplitScan<R> &S, const float (&top)[NS], const unsigned (&sum)[NS],
                                                     const unsigned (&cnt)[NS]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int row, q, half;
            coords(u, row, q, half);
#pragma unroll
            for (int c = 0; c < NS / U; ++c) {
                const int i = u * (NS / U) + c;
                atomicMax(&S.top[row + c], __float_as_uint(top[i]));
                atomicAdd(&S.sum[row + c], sum[i]);
                atomicAdd(&S.cnt[row + c], cnt[i]);
            }
        }
    }
    // unit u's values scaled, split and written
    static __device__ __forceinline__ void store(char *H, char *L, const f4v_t (&reg)[NF], const float (&sc)[NS], int u) {
        int row, q, half;
        coords(u, row, q, half);
        if (KC) {
            h8v_t h, l;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                h2v_t a, b;
                const f4v_t &v = reg[2 * u + e / 4];
                split2(v[e & 3], sc[u], v[(e & 3) + 1], sc[u], a, b);
                h[e] = a[0];
                h[e + 1] = a[1];
                l[e] = b[0];
                l[e + 1] = b[1];
            }
            const int to = at(row, q);
            *reinterpret_cast<h8v_t *>(H + to) = h;
            *reinterpret_cast<h8v_t *>(L + to) = l;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                h4v_t h, l;
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    h2v_t a, b;
                    split2(reg[4 * u + e][c], sc[4 * u + c], reg[4 * u + e + 1][c], sc[4 * u + c], a, b);
                    h[e] = a[0];
                    h[e + 1] = a[1];
                    l[e] = b[0];
                    l[e + 1] = b[1];
                }
                const int to = at(row, q) + c % (G / 16) * 1024 + c / (G / 16) * 16 + 8 * half;
                *reinterpret_cast<h4v_t *>(H + to) = h;
                *reinterpret_cast<h4v_t *>(L + to) = l;
            }
        }
    }
};

// The scale exponents of R rows (into S.top, as int), and whether the tile has
// one that cannot be split.
template <int R, int NT>
__device__ __forceinline__ void split_scales(SplitScan<R> &S, int *bad) {
    for (int r = threadIdx.x; r < R; r += NT) {
        const int e = static_cast<int>(S.top[r] >> 23), n = static_cast<int>(S.cnt[r]);
        const int mean = n ? static_cast<int>(S.sum[r] / n) : e;
        if (S.top[r] != 0 && (e == 255 || e < kSplitTopExp - 127 || e - mean > kSplitSpread)) *bad = 1;
        S.top[r] = static_cast<unsigned>(S.top[r] != 0 ? kSplitTopExp - e : 0);
    }
}

// ---- the scan as a launch of its own -------------------------------------------------
//
// Where the caller's workspace has room, the operands are scanned once, before
// the product, instead of by every workgroup: per slice of K, row and chunk of
// k one SplitRow, the chunks' exact sums added up by the product's workgroups
// (the same scales and choices as their own scan, and so the same bits).
// HBM-bound: each operand read once (40 us for 8192 x 4096 and 4096 x 4096).
struct SplitRow {
    unsigned top, sum, cnt, pad;
};
constexpr int kScanRows = 16;    // k-contiguous: rows per workgroup, four per wave
constexpr int kScanCols = 64;    // else: columns per workgroup, four per lane, 16 k side by side
constexpr int kScanChunks = 16;  // at most this many chunks of k
struct SplitScanArgs {
    SplitRow *a, *b;             // [slice][chunk][row]; null a: no scan
    int chunks_a, chunks_b, kc_a, kc_b;  // chunks of k (per slice), and k per chunk
    int blocks_a, blocks_b;      // workgroups per slice
};

__device__ __forceinline__ void scan_value(float v, unsigned &top, unsigned &sum, unsigned &cnt) {
    const unsigned e = __builtin_amdgcn_ubfe(__float_as_uint(v), 23, 8);
    top = __float_as_uint(fmaxf(__uint_as_float(top), fabsf(v)));
    sum += e;
    cnt += min(e, 1u);
}

template <bool XF>
__device__ __forceinline__ f4v_t scan_load(const float *p, int have, const XfRegs &xf) {
    f4v_t v[1];
    if (have >= 4) v[0] = *reinterpret_cast<const f4u_t *>(p);
    else v[0] = f4v_t{p[0], have > 1 ? p[1] : 0.0f, have > 2 ? p[2] : 0.0f, 0.0f};
    if constexpr (XF) xf_regs(xf, v);
    return v[0];
}

// Rows of a k-contiguous operand: a wave takes four, 256 k of each at a time.
template <bool XF>
__device__ __forceinline__ void scan_rows(const float *X, int rows, int K, int ld, SplitRow *out, int block,
                                          const XfRegs &xf) {
    const int lane = threadIdx.x & 63, r0 = block * kScanRows + static_cast<int>(threadIdx.x >> 6) * 4;
    unsigned top[4] = {}, sum[4] = {}, cnt[4] = {};
#pragma unroll 2
    for (int k = lane * 4; k < K; k += 256) {
        f4v_t v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = scan_load<XF>(X + (size_t)min(r0 + r, rows - 1) * ld + k, K - k, xf);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) scan_value(v[r][c], top[r], sum[r], cnt[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            top[r] = max(top[r], (unsigned)__shfl_xor((int)top[r], d, 64));
            sum[r] += __shfl_xor((int)sum[r], d, 64);
            cnt[r] += __shfl_xor((int)cnt[r], d, 64);
        }
        if (lane == r && r0 + r < rows) out[r0 + r] = SplitRow{top[r], sum[r], cnt[r], 0};
    }
}

// Columns of the other kind over one chunk of k: 16 lanes take four each, the
// workgroup's 16 groups of lanes every 16th k.
template <bool XF>
__device__ __forceinline__ void scan_cols(const float *X, int rows, int K, int ld, SplitRow *out, int block,
                                          int chunks, int kc, const XfRegs &xf) {
    __shared__ unsigned part[3][16][kScanCols];  // top, sum, cnt
    const int t = threadIdx.x, cl = (t & 15) * 4, kp = t >> 4;
    const int chunk = block % chunks, c0 = (block / chunks) * kScanCols;
    const int k1 = min(K, (chunk + 1) * kc), have = rows - c0 - cl;
    unsigned top[4] = {}, sum[4] = {}, cnt[4] = {};
    if (have > 0) {
#pragma unroll 4
        for (int k = chunk * kc + kp; k < k1; k += 16) {
            const f4v_t v = scan_load<XF>(X + (size_t)k * ld + c0 + cl, have, xf);
#pragma unroll
            for (int c = 0; c < 4; ++c) scan_value(v[c], top[c], sum[c], cnt[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        part[0][kp][cl + c] = top[c];
        part[1][kp][cl + c] = sum[c];
        part[2][kp][cl + c] = cnt[c];
    }
    __syncthreads();
    if (t < kScanCols && c0 + t < rows) {
        SplitRow r{0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            r.top = max(r.top, part[0][w][t]);
            r.sum += part[1][w][t];
            r.cnt += part[2][w][t];
        }
        out[(size_t)chunk * rows + c0 + t] = r;
    }
}

template <bool TA, bool TB, bool XF>
__global__ __launch_bounds__(256) void split_scan(GemmArgs g, SplitScanArgs p) {
    const int per = p.blocks_a + p.blocks_b;
    const int slice = static_cast<int>(blockIdx.x) / per;
    int b = static_cast<int>(blockIdx.x) - slice * per;
    const int k0 = slice * g.kslice, K = g.kslice > 0 ? min(g.kslice, g.K - k0) : g.K;
    const XfRegs xf = XF ? xf_load(b < p.blocks_a ? g.xa : g.xb) : XfRegs{};
    if (b < p.blocks_a) {  // uniform
        SplitRow *out = p.a + (size_t)slice * p.chunks_a * g.M;
        const float *X = g.A + (TA ? (size_t)k0 * g.lda : (size_t)k0);
        if constexpr (TA) scan_cols<XF>(X, g.M, K, g.lda, out, b, p.chunks_a, p.kc_a, xf);
        else scan_rows<XF>(X, g.M, K, g.lda, out, b, xf);
    } else {
        b -= p.blocks_a;
        SplitRow *out = p.b + (size_t)slice * p.chunks_b * g.N;
        const float *X = g.B + (TB ? (size_t)k0 : (size_t)k0 * g.ldb);
        if constexpr (TB) scan_rows<XF>(X, g.N, K, g.ldb, out, b, xf);
        else scan_cols<XF>(X, g.N, K, g.ldb, out, b, p.chunks_b, p.kc_b, xf);
    }
}

// R rows from r0 on of a slice's scan into S.
template <int R, int NT>
__device__ __forceinline__ void scan_take(SplitScan<R> &S, const SplitRow *scan, int chunks, int rows, int r0) {
    for (int r = threadIdx.x; r < R; r += NT) {
        const SplitRow *p = scan + min(r0 + r, rows - 1);
        SplitRow v[kScanChunks];  // every load in flight
#pragma unroll
        for (int c = 0; c < kScanChunks; ++c) v[c] = p[(size_t)min(c, chunks - 1) * rows];
        unsigned top = 0, sum = 0, cnt = 0;
#pragma unroll
        for (int c = 0; c < kScanChunks; ++c)
            if (c < chunks) {
                top = max(top, v[c].top);
                sum += v[c].sum;
                cnt += v[c].cnt;
            }
        S.top[r] = top;
        S.sum[r] = sum;
        S.cnt[r] = cnt;
    }
}

template <bool TA, bool TB, int BM, int BN, int WM, int WN, int PF, int EPI, bool CS, bool XF>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split(GemmArgs g, int products, SplitScanArgs scans) {
    constexpr int NT = 64 * WM * WN;
    if (CS && static_cast<int>(blockIdx.x) >= products) {  // uniform: B's column sums, 16 columns a workgroup
        colsum_strip<NT, XF>(g, (static_cast<int>(blockIdx.x) - products) * kStripCols);
        return;
    }
    constexpr int TMW = BM / WM, TNW = BN / WN, FM = TMW / 16, FN = TNW / 16;
    constexpr int GA = !TA ? 16 : TMW >= 64 ? 64 : TMW, GB = TNW >= 64 ? 64 : TNW;
    static_assert(FN == GB / 16, "a wave's columns are one interleave group");
    using SA = SplitStage<BM, GA, NT, !TA>;
    using SB = SplitStage<BN, GB, NT, TB>;
    // h and l of both operands, two stages; the fp32 tile's operands instead
    __shared__ __attribute__((aligned(16))) char lds[2 * (BM + BN) * 128];
    using Half = char(*)[BM * 64];
    using HalfB = char(*)[BN * 64];
    const Half Ah = reinterpret_cast<Half>(lds), Al = Ah + 2;
    const HalfB Bh = reinterpret_cast<HalfB>(lds + BM * 256), Bl = Bh + 2;
    static_assert(2 * (BM + BN) * 128 >= 2 * kBK * 4 * (BM + BN), "room for the fp32 tile");
    __shared__ SplitScan<BM> sa;
    __shared__ SplitScan<BN> sb;
    __shared__ int bad;

    const float *Ap = g.A, *Bp = g.B;
    float *Cp = g.C;
    int bid = blockIdx.x;
    if (g.batch_rank > 0) {
        const int batch = bid / g.tiles;
        bid -= batch * g.tiles;
        long long oa, ob;
        batch_offsets(g, batch, oa, ob);
        Ap += oa;
        Bp += ob;
        Cp += static_cast<long long>(batch) * g.sc;
    }
    int K = g.K, slice = 0;
    if (g.kslice > 0) {  // split K: partial products side by side in C
        slice = bid / g.tiles;
        bid -= slice * g.tiles;
        const int k0 = slice * g.kslice;
        K = min(g.kslice, g.K - k0);
        Ap += TA ? (size_t)k0 * g.lda : (size_t)k0;
        Bp += TB ? (size_t)k0 : (size_t)k0 * g.ldb;
        Cp += (size_t)slice * g.M * g.ldc;
    }
    int tm, tn;
    tile_coords(g.tiles_m, g.tiles_n, bid, tm, tn);
    const int i0 = tm * BM, j0 = tn * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 15, lq = lane >> 4;

    const XfRegs xfa = XF ? xf_load(g.xa) : XfRegs{}, xfb = XF ? xf_load(g.xb) : XfRegs{};
    f4v_t acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[a][b] = f4v_t{0.0f, 0.0f, 0.0f, 0.0f};

    unsigned offa[SA::U], offb[SB::U];
    SA::offsets(offa, g.lda, g.M, i0);
    SB::offsets(offb, g.ldb, g.N, j0);
    const int ai = SA::first(g.M, i0), bj0 = SB::first(g.N, j0);
    const float *Abase = TA ? Ap + ai : Ap + (size_t)ai * g.lda;
    const float *Bbase = TB ? Bp + (size_t)bj0 * g.ldb : Bp + bj0;
    const size_t astep = TA ? (size_t)kSplitK * g.lda : kSplitK, bstep = TB ? kSplitK : (size_t)kSplitK * g.ldb;

    constexpr int UA = SA::U, UB = SB::U, FUA = SA::NF / UA, FUB = SB::NF / UB;
    const int nst = K / kSplitK;  // whole stages, at least one
    f4v_t ra[PF][SA::NF], rb[PF][SB::NF];
    auto load = [&](int slot, int u, int t) {  // unit u (A's, then B's) of stage t
        t = min(t, nst - 1);  // past the end: the last stage again, never used
        if (u < UA) {
#pragma unroll
            for (int f = 0; f < FUA; ++f)
                ra[slot][u * FUA + f] = SA::load(Abase + t * astep, g.lda, offa, u * FUA + f);
        } else {
#pragma unroll
            for (int f = 0; f < FUB; ++f)
                rb[slot][(u - UA) * FUB + f] = SB::load(Bbase + t * bstep, g.ldb, offb, (u - UA) * FUB + f);
        }
    };
    // the scan, or what its own launch found
    const bool edge = (TA && i0 + BM > g.M && (g.M & 3)) || (!TB && j0 + BN > g.N && (g.N & 3));
    const bool tail = nst * kSplitK < K;
    for (int r = threadIdx.x; r < BM; r += NT) sa.top[r] = sa.sum[r] = sa.cnt[r] = 0;
    for (int r = threadIdx.x; r < BN; r += NT) sb.top[r] = sb.sum[r] = sb.cnt[r] = 0;
    if (threadIdx.x == 0) bad = 0;
    if (scans.a) {  // uniform
#pragma unroll
        for (int u = 0; u < UA + UB; ++u) load(0, u, 0);
        __syncthreads();
        scan_take<BM, NT>(sa, scans.a + (size_t)slice * scans.chunks_a * g.M, scans.chunks_a, g.M, i0);
        scan_take<BN, NT>(sb, scans.b + (size_t)slice * scans.chunks_b * g.N, scans.chunks_b, g.N, j0);
        __syncthreads();
    } else {
        float topa[SA::NS] = {}, topb[SB::NS] = {};
        unsigned suma[SA::NS] = {}, sumb[SB::NS] = {}, cnta[SA::NS] = {}, cntb[SB::NS] = {};
        auto scan = [&](f4v_t(&va)[SA::NF], f4v_t(&vb)[SB::NF]) {
            if constexpr (XF) {
                xf_regs(xfa, va);
                xf_regs(xfb, vb);
            }
#pragma unroll
            for (int u = 0; u < UA; ++u) SA::scan(va, u, topa, suma, cnta);
#pragma unroll
            for (int u = 0; u < UB; ++u) SB::scan(vb, u, topb, sumb, cntb);
        };
        constexpr int D = kScanDepth;  // stages in flight
        f4v_t va[D][SA::NF], vb[D][SB::NF];
        auto fetch = [&](int d, int t) {
            t = min(t, nst - 1);  // past the end: the last stage again, not scanned
#pragma unroll
            for (int f = 0; f < SA::NF; ++f) va[d][f] = SA::load(Abase + t * astep, g.lda, offa, f);
#pragma unroll
            for (int f = 0; f < SB::NF; ++f) vb[d][f] = SB::load(Bbase + t * bstep, g.ldb, offb, f);
        };
        auto stages = [&](auto ends) {
            constexpr bool EDGE = decltype(ends)::value;
#pragma unroll
            for (int d = 0; d < D; ++d) fetch(d, d);
            for (int t = 0; t < nst; t += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    if constexpr (EDGE && TA)
                        for (int u = 0; u < UA; ++u) SA::mend(va[d], g.M, i0, u);
                    if constexpr (EDGE && !TB)
                        for (int u = 0; u < UB; ++u) SB::mend(vb[d], g.N, j0, u);
                    if (t + d < nst) scan(va[d], vb[d]);  // uniform
                    fetch(d, t + D + d);
                    __builtin_amdgcn_sched_barrier(0);  // the loads before the next stage is waited for
                }
            }
        };
        if (edge) stages(BoolTag<true>{});
        else stages(BoolTag<false>{});
        if (tail) {
#pragma unroll
            for (int f = 0; f < SA::NF; ++f) va[0][f] = SA::load_edge(Ap, g.lda, g.M, K, i0, nst * kSplitK, f);
#pragma unroll
            for (int f = 0; f < SB::NF; ++f) vb[0][f] = SB::load_edge(Bp, g.ldb, g.N, K, j0, nst * kSplitK, f);
            scan(va[0], vb[0]);
        }
        __syncthreads();
        SA::scan_join(sa, topa, suma, cnta);
        SB::scan_join(sb, topb, sumb, cntb);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < UA + UB; ++u) load(0, u, 0);  // on their way while the scales are found
    }
    split_scales<BM, NT>(sa, &bad);
    split_scales<BN, NT>(sb, &bad);
    __syncthreads();
    if (bad) {  // uniform
        auto Af = reinterpret_cast<float(*)[kBK * BM]>(lds);
        auto Bf = reinterpret_cast<float(*)[kBK * BN]>(lds + 2 * kBK * BM * 4);
        constexpr int FPF = prefetch_tiles<BM>();
        if (g.vec) fp32_tile<TA, TB, BM, BN, WM, WN, EPI, FPF, true, XF>(g, Ap, Bp, Cp, K, i0, j0, Af, Bf);
        else fp32_tile<TA, TB, BM, BN, WM, WN, EPI, FPF, false, XF>(g, Ap, Bp, Cp, K, i0, j0, Af, Bf);
        return;
    }
    float sca[SA::NS], scb[SB::NS];
    SA::scales(sca, sa);
    SB::scales(scb, sb);

    // fragments: block x of an operand's wave tile
    const int fo = (lq * 16 + (li ^ split_x(lq))) * 16;
    auto frag_a = [&](const char *S, int x) { return *reinterpret_cast<const h8v_t *>(S + (wm * FM + x) * 1024 + fo); };
    auto frag_b = [&](const char *S, int x) {
        const int blk = wn * FN + x;
        return *reinterpret_cast<const h8v_t *>(S + blk * 1024 + (SB::kXor ? fo ^ (blk & 3) << 4 : fo));
    };

    h8v_t fah[2], fal[2], fbh[FN], fbl[FN];
    auto read_a = [&](int buf, int x, int slot) {
        fah[slot] = frag_a(Ah[buf], x);
        fal[slot] = frag_a(Al[buf], x);
    };
    auto read_bh = [&](int buf) {
#pragma unroll
        for (int c = 0; c < FN; ++c) fbh[c] = frag_b(Bh[buf], c);
    };
    auto read_bl = [&](int buf) {
#pragma unroll
        for (int c = 0; c < FN; ++c) fbl[c] = frag_b(Bl[buf], c);
    };
    auto mm = [](h8v_t a, h8v_t b, f4v_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); };

    const int flip = max(1, (5 * nst + 4) / 8);  // the first stage of the negated product
    // the loop over whole stages; EDGE: a row-contiguous operand's tile ends
    // inside a float4
    auto whole = [&](auto edge) {
        constexpr bool EDGE = decltype(edge)::value;
        auto put = [&](int buf, int slot, int u) {  // its registers to LDS
            if (u < UA) {
                if constexpr (EDGE && TA) SA::mend(ra[slot], g.M, i0, u);
                if constexpr (XF) {
                    if (u == 0) xf_regs(xfa, ra[slot]);
                }
                SA::store(Ah[buf], Al[buf], ra[slot], sca, u);
            } else {
                if constexpr (EDGE && !TB) SB::mend(rb[slot], g.N, j0, u - UA);
                if constexpr (XF) {
                    if (u == UA) xf_regs(xfb, rb[slot]);
                }
                SB::store(Bh[buf], Bl[buf], rb[slot], scb, u - UA);
            }
        };
#pragma unroll
        for (int u = 0; u < UA + UB; ++u) put(0, 0, u);
#pragma unroll
        for (int s = 0; s < PF; ++s)
#pragma unroll
            for (int u = 0; u < UA + UB; ++u) load(s, u, 1 + s);
        __syncthreads();
        read_a(0, 0, 0);
        read_bh(0);
        read_bl(0);
        for (int t0 = 0; t0 < nst; t0 += PF) {
#pragma unroll
            for (int s = 0; s < PF; ++s) {
                const int t = t0 + s;
                if (PF > 1 && t >= nst) break;  // uniform
                if (t == flip) {  // uniform
#pragma unroll
                    for (int a = 0; a < FM; ++a)
#pragma unroll
                        for (int b = 0; b < FN; ++b) acc[a][b] = -acc[a][b];
                }
                if (t + 1 == flip) {  // stage t + 1 is staged in this one
#pragma unroll
                    for (int i = 0; i < SA::NS; ++i) sca[i] = -sca[i];
                }
                const int cur = t & 1, nxt = cur ^ 1;
#pragma unroll
                for (int x = 0; x < FM; ++x) {
                    constexpr int kSlots = FM - 1;  // the units go over the blocks before the barrier
#pragma unroll
                    for (int u = x * (UA + UB) / kSlots; x < kSlots && u < (x + 1) * (UA + UB) / kSlots; ++u) {
                        put(nxt, s, u);
                        load(s, u, t + 1 + PF);
                    }
                    if (x + 1 < FM) {
                        read_a(cur, x + 1, (x + 1) & 1);
                    } else {
                        __syncthreads();  // stage t + 1 is written; this one's last fragments are in registers
                        read_a(nxt, 0, (x + 1) & 1);
                    }
#pragma unroll
                    for (int c = 0; c < FN; ++c) acc[x][c] = mm(fah[x & 1], fbh[c], acc[x][c]);
#pragma unroll
                    for (int c = 0; c < FN; ++c) acc[x][c] = mm(fal[x & 1], fbh[c], acc[x][c]);
                    if (x + 1 == FM) read_bh(nxt);
#pragma unroll
                    for (int c = 0; c < FN; ++c) acc[x][c] = mm(fah[x & 1], fbl[c], acc[x][c]);
                    if (x + 1 == FM) read_bl(nxt);
                }
            }
        }
    };
    if (edge) whole(BoolTag<true>{});
    else whole(BoolTag<false>{});
    if (tail) {  // a partial last stage
        if (flip == nst) {  // the loop ended at the turn (the scales are negative by now)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] = -acc[a][b];
        }
#pragma unroll
        for (int f = 0; f < SA::NF; ++f) ra[0][f] = SA::load_edge(Ap, g.lda, g.M, K, i0, nst * kSplitK, f);
#pragma unroll
        for (int f = 0; f < SB::NF; ++f) rb[0][f] = SB::load_edge(Bp, g.ldb, g.N, K, j0, nst * kSplitK, f);
        if constexpr (XF) {
            xf_regs(xfa, ra[0]);
            xf_regs(xfb, rb[0]);
        }
        __syncthreads();  // the loop's last reads
#pragma unroll
        for (int u = 0; u < SA::U; ++u) SA::store(Ah[0], Al[0], ra[0], sca, u);
#pragma unroll
        for (int u = 0; u < SB::U; ++u) SB::store(Bh[0], Bl[0], rb[0], scb, u);
        __syncthreads();
        read_bh(0);
        read_bl(0);
#pragma unroll
        for (int x = 0; x < FM; ++x) {
            read_a(0, x, 0);
#pragma unroll
            for (int c = 0; c < FN; ++c) {
                acc[x][c] = mm(fah[0], fbh[c], acc[x][c]);
                acc[x][c] = mm(fal[0], fbh[c], acc[x][c]);
                acc[x][c] = mm(fah[0], fbl[c], acc[x][c]);
            }
        }
    }

    const bool negated = flip < nst || tail;
    // The scales taken back, the epilogue (store_tile's) and the store: lane
    // (li, lq)'s element v of block (x, c) is row i0 + row_of(x, v), column
    // col + c.
    const int col = j0 + wn * TNW + FN * li;
    int ebl[FN];
    float bj[FN];
#pragma unroll
    for (int c = 0; c < FN; ++c) {
        ebl[c] = static_cast<int>(sb.top[wn * TNW + FN * li + c]);
        bj[c] = EPI != kEpiNone && g.bias ? g.bias[min(col + c, g.N - 1)] : 0.0f;
    }
    const bool vec = FN == 4 && (reinterpret_cast<uintptr_t>(Cp) & 15) == 0 && g.ldc % 4 == 0 && col + 3 < g.N &&
                     (EPI != kEpiAll || !g.mask || (reinterpret_cast<uintptr_t>(g.mask) & 15) == 0);
    auto row_of = [&](int x, int v) {
        constexpr int F = GA / 16;
        return wm * TMW + (x / F) * GA + (4 * lq + v) * F + x % F;
    };
#pragma unroll
    for (int x = 0; x < FM; ++x) {
        float mk[4][FN];
        if (EPI == kEpiAll && g.mask) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const size_t at = (size_t)min(i0 + row_of(x, v), g.M - 1) * g.ldc;
                if (vec) {
                    const f4v_t m = *reinterpret_cast<const f4v_t *>(g.mask + at + col);
#pragma unroll
                    for (int c = 0; c < FN; ++c) mk[v][c] = m[c];
                } else {
#pragma unroll
                    for (int c = 0; c < FN; ++c) mk[v][c] = g.mask[at + min(col + c, g.N - 1)];
                }
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = row_of(x, v), er = static_cast<int>(sa.top[r]);
            float o[FN];
#pragma unroll
            for (int c = 0; c < FN; ++c) {
                float val = __builtin_ldexpf(negated ? -acc[x][c][v] : acc[x][c][v], -(er + ebl[c]));
                if (EPI != kEpiNone) {
                    if (g.bias) val = val + bj[c];
                    if (g.relu) val = val > 0.0f ? val : 0.0f;
                    if (EPI == kEpiAll && g.mask) val = mk[v][c] > 0.0f ? val : 0.0f;
                }
                o[c] = val;
            }
            if (i0 + r < g.M) {
                float *q = Cp + (size_t)(i0 + r) * g.ldc + col;
                if (vec) {
                    if constexpr (FN == 4) *reinterpret_cast<f4v_t *>(q) = f4v_t{o[0], o[1], o[2], o[3]};
                } else {
#pragma unroll
                    for (int c = 0; c < FN; ++c)
                        if (col + c < g.N) q[c] = o[c];
                }
            }
        }
    }
}

// The slices' partial products (row pitch ldp, a multiple of 4) added in slice
// order, with the epilogue: a thread takes four columns of a row, a workgroup
// 256 columns of four rows.  HBM-bound (the partials from the caches): a
// division per element to find its row made it 28 us for 4 x 1003 x 2050.
constexpr int kSplitMaxSlices = 16;
__global__ __launch_bounds__(256) void split_sum(const float *__restrict__ P, int slices, int ldp, GemmArgs g) {
    const int col = (static_cast<int>(blockIdx.x) * 64 + static_cast<int>(threadIdx.x & 63)) * 4;
    const int row = static_cast<int>(blockIdx.y) * 4 + static_cast<int>(threadIdx.x >> 6);
    if (row >= g.M || col >= g.N) return;
    const size_t plane = static_cast<size_t>(g.M) * ldp, at = static_cast<size_t>(row) * ldp + col;
    f4v_t v[kSplitMaxSlices];  // every slice in flight
#pragma unroll
    for (int k = 0; k < kSplitMaxSlices; ++k)
        if (k < slices) v[k] = *reinterpret_cast<const f4v_t *>(P + k * plane + at);
    f4v_t acc = v[0];
#pragma unroll
    for (int k = 1; k < kSplitMaxSlices; ++k)
        if (k < slices) acc += v[k];
    const size_t to = static_cast<size_t>(row) * g.ldc + col;
    const bool vec = col + 3 < g.N && (reinterpret_cast<uintptr_t>(g.C + to) & 15) == 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int j = min(col + c, g.N - 1);
        float x = acc[c];
        if (g.bias) x = x + g.bias[j];
        if (g.relu) x = x > 0.0f ? x : 0.0f;
        if (g.mask) x = g.mask[static_cast<size_t>(row) * g.ldc + j] > 0.0f ? x : 0.0f;
        acc[c] = x;
    }
    if (vec) {
        *reinterpret_cast<f4v_t *>(g.C + to) = acc;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (col + c < g.N) g.C[to + c] = acc[c];
    }
}

}  // namespace tship
