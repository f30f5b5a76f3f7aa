// fp32 products on the bf16 matrix cores (the kernels; ts_hip_gemm_split.hip
// chooses and launches them).
//
// The fp32 matrix instructions bound the large products at 157 TFLOP/s; the
// bf16 ones run 16 times as fast.  Every fp32 value is exactly the sum of three
// bf16 values, each the rounding of what the ones before leave:
//   h = bf16(v), m = bf16(v - h), l = v - h - m   (8 significant bits each),
// with |m| <= 2^-8 |v| and |l| <= 2^-17 |v|, so of the nine products of the
// pieces of a and b the six down to 2^-16 |a b| are summed in fp32,
//   a b = ha hb + (ha mb + ma hb) + (ma mb + ha lb + la hb),
// and the three left out are below 2^-24 |a b| together: less than one rounding
// of the term.  bf16 has fp32's exponents, so this holds for every value
// whatever else its row holds; there is no common scale.
//
// Range.  Both operands are staged times 2^16 (exact) and the finished sums
// taken back by 2^-32 (ldexp, one rounding): the pieces of the smallest
// subnormals are then bf16 values too.  A NaN is NaN in h, and so in the sums it
// enters.  Where a sum is not finite for another reason -- an infinity in an
// operand, a value past 2^111 or a sum past 2^95 -- the tile is computed again on
// the fp32 instructions (fp32_tile) and has their result.
//
// Sums.  Six instructions add up the pieces' products of 16 k from zero, and the
// vector units add that to the running sum, so it is rounded once per 16 k
// (the fp32 instructions: per 2 k).  The matrix instruction drops the lowest bits
// of its sum downwards, the same way in every element and call; so every second
// stage is of the negated product, subtracted, and the two errors cancel.
// Error against 64 bits, fp32 instructions and these, of normal data: K = 1024
// 5.7e-7, 1.3e-7 to 1.6e-7; K = 4096 1.15e-6, 2.2e-7; with four fifths of B zero
// 2.5e-7, 1.3e-7.  (Summed straight into the running sum: 4.9e-7, 9.8e-7, 4.0e-7.)
//
// Tiles.  BM x BN per workgroup in LDS stages of 16 k, two of them.  A stage's
// global loads are issued NH stages before they are scaled, split and written to
// LDS, which happens while the fragments of the stage before feed the matrix
// cores; one barrier per stage, before its last row of blocks so that their
// MFMAs cover the first reads of the next.  KG groups of waves each take a part
// of K.  Bound by the vector units (splitting and adding) as much as by the
// matrix cores: NT 8192 x 4096 x 4096 1435 us (1868 on the fp32 instructions), 192
// TFLOP/s; TN 4096 x 4096 x 8192 1454 (1850); 64 x NN 1024 x 128 x 1024 112 (246).
//
// LDS.  A piece of an operand's stage is [row block of 32][64 chunks of 16
// bytes], a chunk holding eight k of a row (at()); a fragment (row i, k half)
// is one 16-byte read.  Rows are interleaved over the wave tile's F blocks (row
// i * F + b in block b), so a lane owns neighbouring columns of C, and four rows
// of a row-contiguous operand's float4 go to as many blocks.  The chunk is XORed
// with bits of the half, the block and i >> 3 so that the writes of a group of
// lanes fall in different banks; reads stay within aligned groups of eight
// chunks, in any order free of conflicts.
#pragma once

#include "ts_hip_gemm_common.h"

typedef __bf16 b2v_t __attribute__((ext_vector_type(2)));
typedef __bf16 b8v_t __attribute__((ext_vector_type(8)));
typedef float f2v_t __attribute__((ext_vector_type(2)));
typedef float f2u_t __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned u2v_t __attribute__((ext_vector_type(2)));
// four floats at any 4-byte address (gfx950 loads them with one instruction)
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

namespace tship {

constexpr int kSplitK = 16;  // k of a stage
constexpr float kSplitScale = 65536.0f;
constexpr int kSplitScaleExp = 32;  // of a product

// ---- staging ----------------------------------------------------------------------

// two values times s as their three pieces
struct Pieces {
    unsigned h, m, l;  // two bf16 each
};
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    const f2v_t v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, b2v_t));
}
__device__ __forceinline__ Pieces split2(float a, float b, float s) {
    auto low = [](unsigned p) { return __uint_as_float(p << 16); };
    auto high = [](unsigned p) { return __uint_as_float(p & 0xffff0000u); };
    Pieces p;
    a *= s;
    b *= s;
    p.h = bf16_pair(a, b);
    a -= low(p.h);
    b -= high(p.h);
    p.m = bf16_pair(a, b);
    p.l = bf16_pair(a - low(p.m), b - high(p.m));
    return p;
}

// One operand's staging by NT threads: R rows in groups of 32 F interleaved
// over F blocks, 16 k at a time.
// KC (k contiguous): a thread's unit is one row and a quarter of the k (one
// float4); else four rows and two k (two float4, four rows each).
template <int R, int F, int NT, bool KC>
struct SplitStage {
    static constexpr int kUnits = KC ? R * 4 : R * 2;
    static constexpr int U = (kUnits + NT - 1) / NT;  // units per thread
    static constexpr int NF = KC ? U : 2 * U;         // float4 per thread
    static_assert((kUnits % NT == 0 || NT % kUnits == 0) && (KC || U == 1) && F <= 2, "units");
    static constexpr int kPiece = R * 2 * kSplitK;  // bytes of one piece of a stage
    static constexpr int kStage = 3 * kPiece;

    // byte address, within a piece, of row `row` and half `half` of a stage's k
    static __device__ __forceinline__ int at(int row, int half) {
        const int blk = row / (32 * F) * F + row % F, i = row % (32 * F) / F;
        return blk * 1024 + ((half * 32 + i) ^ mix(blk, half, i)) * 16;
    }
    static __device__ __forceinline__ int mix(int blk, int half, int i) {
        if (!KC) return F == 2 ? i >> 3 & 1 : i >> 3 & 3;
        return F == 2 ? 6 * (blk & 1) ^ 10 * half : 12 * half;
    }
    // a thread's first unit: its (first) row, and its part of a stage's k: KC a
    // quarter, else a pair (the next unit's row: NT / 4 on)
    static __device__ __forceinline__ void coords(int thread, int &row, int &part) {
        const int n = thread % kUnits;
        if (KC) {
            row = n >> 2;
            part = n & 3;
        } else {  // four neighbouring lanes fill a chunk
            row = 4 * ((n >> 2) % (R / 4));
            part = (n & 3) + 4 * (n / R);
        }
    }
    // byte offset of a thread's first float4 from the tile's first row and the stage's first k
    static __device__ __forceinline__ unsigned offset(int thread, int ld) {
        int row, part;
        coords(thread, row, part);
        const unsigned pitch = 4u * static_cast<unsigned>(ld);
        return KC ? static_cast<unsigned>(row) * pitch + 16u * part : 2u * part * pitch + 4u * row;
    }
    // float4 number f of a whole stage
    static __device__ __forceinline__ f4v_t load(const float *base, int ld, unsigned off, int f) {
        const char *p = reinterpret_cast<const char *>(base + (size_t)(KC ? f * (NT / 4) : f) * ld);
        return *reinterpret_cast<const f4u_t *>(p + off);
    }
    // the same at k0, zeros from K on
    static __device__ __forceinline__ f4v_t load_edge(const float *base, int thread, int ld, int k0, int K, int f) {
        int row, part;
        coords(thread, row, part);
        f4v_t v;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int r = KC ? row + f * (NT / 4) : row + c, k = k0 + (KC ? 4 * part + c : 2 * part + f);
            const size_t kk = min(k, K - 1);
            const float x = KC ? base[(size_t)r * ld + kk] : base[kk * ld + r];
            v[c] = k < K ? x : 0.0f;
        }
        return v;
    }
    // the largest magnitude among a thread's values of the tile's rows (NaNs aside)
    template <bool XF>
    static __device__ __forceinline__ float largest(const float *base, int thread, int ld, size_t step, int K,
                                                    const XfRegs &xf) {
        const unsigned off = offset(thread, ld);
        float m = 0.0f;
        auto take = [&](f4v_t (&v)[NF]) {
            if constexpr (XF) xf_regs(xf, v);
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int c = 0; c < 4; ++c) m = fmaxf(m, fabsf(v[f][c]));
        };
        int k = 0;
#pragma unroll 4
        for (; k + kSplitK <= K; k += kSplitK, base += step) {
            f4v_t v[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) v[f] = load(base, ld, off, f);
            take(v);
        }
        if (k < K) {
            f4v_t v[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) v[f] = load_edge(base, thread, ld, 0, K - k, f);
            take(v);
        }
        return m;
    }
    // unit u's values times sc, split, into a stage
    static __device__ __forceinline__ void store(char *S, int thread, const f4v_t (&reg)[NF], float sc, int u) {
        int row, part;
        coords(thread, row, part);
        if (KC) {
            const f4v_t &v = reg[u];
            const Pieces a = split2(v[0], v[1], sc), b = split2(v[2], v[3], sc);
            char *to = S + at(row + u * (NT / 4), part >> 1) + 8 * (part & 1);
            *reinterpret_cast<u2v_t *>(to) = u2v_t{a.h, b.h};
            *reinterpret_cast<u2v_t *>(to + kPiece) = u2v_t{a.m, b.m};
            *reinterpret_cast<u2v_t *>(to + 2 * kPiece) = u2v_t{a.l, b.l};
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const Pieces a = split2(reg[0][c], reg[1][c], sc);
                char *to = S + at(row + c, part >> 2) + 4 * (part & 3);
                *reinterpret_cast<unsigned *>(to) = a.h;
                *reinterpret_cast<unsigned *>(to + kPiece) = a.m;
                *reinterpret_cast<unsigned *>(to + 2 * kPiece) = a.l;
            }
        }
    }
};

// KG groups of WM x WN waves share a tile, each with a part of K and LDS stages
// of its own; their sums are added in order.  NH: stages of loads in flight.
template <bool TA, bool TB, int BM, int BN, int WM, int WN, int KG, int NH, int EPI, bool CS, bool XF>
__global__ __launch_bounds__(64 * WM * WN * KG, KG > 2 ? KG : 2) void gemm_split(GemmArgs g, int products) {
    constexpr int NT = 64 * WM * WN;
    if (CS && static_cast<int>(blockIdx.x) >= products) {  // uniform: B's column sums, 16 columns a workgroup
        colsum_strip<NT * KG, XF>(g, (static_cast<int>(blockIdx.x) - products) * kStripCols);
        return;
    }
    constexpr int TMW = BM / WM, TNW = BN / WN, FM = TMW / 32, FN = TNW / 32;
    using SA = SplitStage<BM, FM, NT, !TA>;
    using SB = SplitStage<BN, FN, NT, TB>;
    // two stages of both operands for each group; the groups' sums, and the
    // fp32 tile's operands, instead
    constexpr int kGroupLds = 2 * (SA::kStage + SB::kStage);
    __shared__ __attribute__((aligned(16))) char lds[KG * kGroupLds];
    static_assert(KG * kGroupLds >= (KG - 1) * BM * BN * 4, "room for the groups' sums");
    __shared__ int bad;
    __shared__ unsigned top[2];

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
    int tm, tn;
    tile_coords(g.tiles_m, g.tiles_n, bid, tm, tn);
    // The last tile of a row or column of tiles ends with the operand (M >= BM,
    // N >= BN): it computes some of its neighbour's rows too and stores only its own.
    const int im = tm * BM, jn = tn * BN, i0 = min(im, g.M - BM), j0 = min(jn, g.N - BN);
    const int lane = threadIdx.x & 63, any_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = KG > 1 ? any_wave / (WM * WN) : 0, wave = KG > 1 ? any_wave % (WM * WN) : any_wave;
    const int thread = static_cast<int>(threadIdx.x) - group * NT;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 31, lh = lane >> 5;
    auto stage_a = [&](int buf) { return lds + group * kGroupLds + buf * SA::kStage; };
    auto stage_b = [&](int buf) { return lds + group * kGroupLds + 2 * SA::kStage + buf * SB::kStage; };

    const XfRegs xfa = XF ? xf_load(g.xa) : XfRegs{}, xfb = XF ? xf_load(g.xb) : XfRegs{};
    float acc[FM][FN][16];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    const unsigned offa = SA::offset(thread, g.lda), offb = SB::offset(thread, g.ldb);
    const float *At = TA ? Ap + i0 : Ap + (size_t)i0 * g.lda, *Bt = TB ? Bp + (size_t)j0 * g.ldb : Bp + j0;
    const size_t astep = TA ? (size_t)kSplitK * g.lda : kSplitK, bstep = TB ? kSplitK : (size_t)kSplitK * g.ldb;

    // the whole stages of K, an even number; this group's: `per` (even) from
    // `from` on (past the last: zeros)
    const int stages = g.K / (2 * kSplitK) * 2;
    const int per = KG > 1 ? (stages / 2 + KG - 1) / KG * 2 : stages, from = group * per;
    // an operand of fewer units than threads: A's are the first waves', B's the last waves'
    const bool has_a = SA::kUnits >= NT || wave < SA::kUnits / 64;
    const bool has_b = SB::kUnits >= NT || wave >= (NT - SB::kUnits) / 64;
    f4v_t ra[NH][SA::NF], rb[NH][SB::NF];
    auto load = [&](int slot, int h) {  // stage h's values (past the end: the last one's again, not used)
        const int at = min(from + h, stages - 1);
        if (has_a) {
#pragma unroll
            for (int f = 0; f < SA::NF; ++f) ra[slot][f] = SA::load(At + at * astep, g.lda, offa, f);
        }
        if (has_b) {
#pragma unroll
            for (int f = 0; f < SB::NF; ++f) rb[slot][f] = SB::load(Bt + at * bstep, g.ldb, offb, f);
        }
    };
    auto ready = [&](int slot) {  // a stage's values as they go to LDS
        if constexpr (XF) {
            xf_regs(xfa, ra[slot]);
            xf_regs(xfb, rb[slot]);
        }
    };
    constexpr int UA = SA::U, UB = SB::U;
    auto put = [&](int buf, int slot, float sc, int u) {  // unit u (A's, then B's) to LDS
        if (u < UA) {
            if (has_a) SA::store(stage_a(buf), thread, ra[slot], sc, u);
        } else if (has_b) {
            SB::store(stage_b(buf), thread, rb[slot], kSplitScale, u - UA);
        }
    };
    // stage h's scale of A: every second stage is of the negated product
    auto scale = [&](int h) { return KG > 1 && from + h >= stages ? 0.0f : h & 1 ? -kSplitScale : kSplitScale; };

    // fragments: block x of an operand's wave tile, piece p
    auto frag = [&](const char *S, int piece, int blk, int mix) {
        return *reinterpret_cast<const b8v_t *>(S + piece + blk * 1024 + ((lh * 32 + li) ^ mix) * 16);
    };
    b8v_t fa[3], fb[FN][3];
    auto read_a = [&](int buf, int x, int p) {
        fa[p] = frag(stage_a(buf), p * SA::kPiece, wm * FM + x, SA::mix(x, lh, li));
    };
    auto read_b = [&](int buf, int c) {
#pragma unroll
        for (int p = 0; p < 3; ++p) fb[c][p] = frag(stage_b(buf), p * SB::kPiece, wn * FN + c, SB::mix(c, lh, li));
    };
    // The pieces' products of block (x, c), summed from zero; A's pieces are
    // replaced by those of block nx of stage `buf` as they fall free (nx < 0: they
    // stay).  The sum joins acc a block later, beside that one's products (minus:
    // the one that joins now is of a negated stage).
    floatx16 sum = {};
    auto join = [&](int n, bool minus) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float &v = acc[n / FN][n % FN][r];
            v = minus ? v - sum[r] : v + sum[r];
        }
    };
    auto block = [&](int n, int buf, int nx, bool minus) {
        const int c = n % FN;
        auto mm = [&](floatx16 s, int pa, int pb) {
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[pa], fb[c][pb], s, 0, 0, 0);
        };
        floatx16 s = {};
        s = mm(s, 0, 2);
        s = mm(s, 0, 1);
        s = mm(s, 0, 0);
        if (nx >= 0) read_a(buf, nx, 0);
        s = mm(s, 1, 1);
        s = mm(s, 1, 0);
        if (nx >= 0) read_a(buf, nx, 1);
        s = mm(s, 2, 0);
        if (nx >= 0) read_a(buf, nx, 2);
        join((n + FM * FN - 1) % (FM * FN), minus);
        sum = s;
    };

    if (threadIdx.x == 0) bad = 0;
#pragma unroll
    for (int h = 0; h < NH; ++h) load(h, h);
    ready(0);
#pragma unroll
    for (int u = 0; u < UA + UB; ++u) put(0, 0, scale(0), u);
    load(0, NH);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 3; ++p) read_a(0, 0, p);
#pragma unroll
    for (int c = 0; c < FN; ++c) read_b(0, c);
    constexpr int N = NH > 2 ? NH : 2;
    static_assert(N % 2 == 0, "stages in pairs");
    for (int h0 = 0; h0 < per; h0 += N) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int h = h0 + i;
            if (N > 2 && h >= per) break;  // uniform
            // stage h's products, and stage h + 1 from the registers to LDS
            const int cur = i & 1, nxt = cur ^ 1, rs = (i + 1) % NH;
            const float sc = scale(h + 1);
            ready(rs);
            // the units go over the blocks before the barrier, which comes before the last row of blocks
            constexpr int kSlots = FM > 1 ? (FM - 1) * FN : 1;
#pragma unroll
            for (int n = 0; n < FM * FN; ++n) {
                const int x = n / FN, c = n % FN;
#pragma unroll
                for (int u = n * (UA + UB) / kSlots; n < kSlots && u < (n + 1) * (UA + UB) / kSlots; ++u)
                    put(nxt, rs, sc, u);
                if (n == kSlots - 1) load(rs, h + 1 + NH);
                if (n == (FM - 1) * FN) __syncthreads();  // the next stage is written, this one read
                block(n, x + 1 == FM ? nxt : cur, c + 1 < FN ? -1 : x + 1 == FM ? 0 : x + 1, (n == 0) != (cur == 1));
                if (x + 1 == FM) read_b(nxt, c);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    join(FM * FN - 1, true);
    sum = floatx16{};
    if (stages * kSplitK < g.K) {  // a partial pair of stages (the first group keeps it)
        const float sc = group == 0 ? kSplitScale : 0.0f;
#pragma unroll 1
        for (int k0 = stages * kSplitK; k0 < g.K; k0 += kSplitK) {
            if (has_a) {
#pragma unroll
                for (int f = 0; f < SA::NF; ++f) ra[0][f] = SA::load_edge(At, thread, g.lda, k0, g.K, f);
            }
            if (has_b) {
#pragma unroll
                for (int f = 0; f < SB::NF; ++f) rb[0][f] = SB::load_edge(Bt, thread, g.ldb, k0, g.K, f);
            }
            ready(0);
            __syncthreads();  // the last reads
#pragma unroll
            for (int u = 0; u < UA + UB; ++u) put(0, 0, sc, u);
            __syncthreads();
#pragma unroll
            for (int p = 0; p < 3; ++p) read_a(0, 0, p);
#pragma unroll
            for (int c = 0; c < FN; ++c) read_b(0, c);
#pragma unroll
            for (int n = 0; n < FM * FN; ++n) block(n, 0, n % FN + 1 < FN ? -1 : (n / FN + 1) % FM, false);
        }
    }
    join(FM * FN - 1, false);

    if constexpr (KG > 1) {  // the other groups' sums, in order
        float *const sums = reinterpret_cast<float *>(lds);
        __syncthreads();  // the last reads
        if (group > 0) {
#pragma unroll
            for (int n = 0; n < FM * FN; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    sums[(((group - 1) * FM * FN + n) * 16 + r) * NT + thread] = acc[n / FN][n % FN][r];
        }
        __syncthreads();
        if (group > 0) return;  // the barriers to come wait for the waves that are left
#pragma unroll 1
        for (int k = 0; k < KG - 1; ++k)
#pragma unroll
            for (int n = 0; n < FM * FN; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n / FN][n % FN][r] += sums[((k * FM * FN + n) * 16 + r) * NT + thread];
    }

    // A sum that is not finite: it stays if it can only be a NaN of the operands'
    // (their finite values too small for a sum to pass the range), else the tile
    // again on the fp32 instructions.
    {
        float worst = 0.0f;  // NaN * 0 and inf * 0 stay NaN
#pragma unroll
        for (int n = 0; n < FM * FN; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) worst = __builtin_fmaf(acc[n / FN][n % FN][r], 0.0f, worst);
        if (worst != worst) bad = 1;
        __syncthreads();
        if (bad) {  // uniform
            if (thread < 2) top[thread] = 0;
            __syncthreads();
            if (has_a) atomicMax(&top[0], __float_as_uint(SA::template largest<XF>(At, thread, g.lda, astep, g.K, xfa)));
            if (has_b) atomicMax(&top[1], __float_as_uint(SB::template largest<XF>(Bt, thread, g.ldb, bstep, g.K, xfb)));
            __syncthreads();
            if (static_cast<double>(__uint_as_float(top[0])) * __uint_as_float(top[1]) * g.K >= 0x1p94 ||
                !(__uint_as_float(top[0]) < 0x1p111f && __uint_as_float(top[1]) < 0x1p111f)) {
                static_assert(KG * kGroupLds >= 2 * kBK * 4 * (BM + BN), "room for the fp32 tile");
                auto Af = reinterpret_cast<float(*)[kBK * BM]>(lds);
                auto Bf = reinterpret_cast<float(*)[kBK * BN]>(lds + 2 * kBK * BM * 4);
                fp32_tile<TA, TB, BM, BN, WM, WN, EPI, 1, false, XF>(g, Ap, Bp, Cp, g.K, im, jn, Af, Bf);
                return;
            }
        }
    }

    // The scale taken back, the epilogue (store_tile's) and the store: lane
    // (li, lh)'s register r of block (x, c) is row row_of(x, r), column col + c.
    const int col = j0 + wn * TNW + FN * li;
    float bj[FN];
#pragma unroll
    for (int c = 0; c < FN; ++c) bj[c] = EPI != kEpiNone && g.bias ? g.bias[col + c] : 0.0f;
    auto row_of = [&](int x, int r) { return i0 + wm * TMW + (8 * (r >> 2) + 4 * lh + (r & 3)) * FM + x; };
#pragma unroll
    for (int x = 0; x < FM; ++x) {
        float mk[16][FN];
        if (EPI == kEpiAll && g.mask) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float *m = g.mask + (size_t)row_of(x, r) * g.ldc + col;
                if constexpr (FN == 2) {
                    const f2v_t v = *reinterpret_cast<const f2u_t *>(m);
                    mk[r][0] = v[0];
                    mk[r][1] = v[1];
                } else {
                    mk[r][0] = m[0];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float o[FN];
#pragma unroll
            for (int c = 0; c < FN; ++c) {
                float val = __builtin_ldexpf(acc[x][c][r], -kSplitScaleExp);
                if (EPI != kEpiNone) {
                    if (g.bias) val = val + bj[c];
                    if (g.relu) val = val > 0.0f ? val : 0.0f;
                    if (EPI == kEpiAll && g.mask) val = mk[r][c] > 0.0f ? val : 0.0f;
                }
                o[c] = val;
            }
            const int row = row_of(x, r);
            if (row < im) continue;  // the neighbour's
            float *q = Cp + (size_t)row * g.ldc + col;
            if (FN == 2 && col >= jn) {
                *reinterpret_cast<f2u_t *>(q) = f2u_t{o[0], o[FN - 1]};
            } else {
#pragma unroll
                for (int c = 0; c < FN; ++c)
                    if (col + c >= jn) q[c] = o[c];
            }
        }
    }
}

}  // namespace tship
