// softmax along one axis (tensor/ops/softmax.rs:4-60) and its backward
// (grad_fn/ops/softmax.rs:4-38).  The tensor is viewed as [outer, reduce,
// inner]; a slice's `reduce` elements are taken in the reference's order --
// max, then exp and a sequential fp32 sum, then a scale by 1/sum; backward a
// sequential fp32 dot then y * (go - dot) -- so the results are those of the
// reference's loops, element for element.
//
// Three forms.  Slices along the last axis (inner == 1) are rows of memory:
// softmax_rows_* hold them in registers, a wave reading and writing 64
// consecutive floats, and only the additions whose order is fixed run one
// after another; many long rows stream through softmax_long_*.  Other axes, and
// rows too short for that, take a thread per slice (softmax_fwd / softmax_bwd),
// whose loads are consecutive along `inner`.
#include "ts_hip_internal.h"
#include "ts_hip_libm.h"

namespace tship {

// f32::exp of the reference: the host libm's expf, restated (ts_hip_libm.h)
__device__ inline float softmax_exp(float x) { return libm::expf_glibc(x); }

__global__ __launch_bounds__(kBlock) void softmax_fwd(const float *__restrict__ x, float *__restrict__ y,
                                                      size_t outer, size_t reduce, size_t inner) {
    const size_t slices = outer * inner;
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t t = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; t < slices; t += stride) {
        const size_t o = t / inner, i = t % inner;
        const size_t base = o * reduce * inner + i;
        float maxv = -__builtin_inff();
        for (size_t j = 0; j < reduce; ++j) {
            const float v = x[base + j * inner];
            if (v > maxv) maxv = v;
        }
        float sum = 0.0f;
        for (size_t j = 0; j < reduce; ++j) {
            const float e = softmax_exp(x[base + j * inner] - maxv);
            y[base + j * inner] = e;
            sum += e;
        }
        const float inv = 1.0f / sum;
        for (size_t j = 0; j < reduce; ++j) y[base + j * inner] *= inv;
    }
}

__global__ __launch_bounds__(kBlock) void softmax_bwd(const float *__restrict__ y, const float *__restrict__ go,
                                                      float *__restrict__ gi, size_t outer, size_t reduce,
                                                      size_t inner) {
    const size_t slices = outer * inner;
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t t = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; t < slices; t += stride) {
        const size_t o = t / inner, i = t % inner;
        const size_t base = o * reduce * inner + i;
        float dot = 0.0f;
        for (size_t j = 0; j < reduce; ++j) {
            const size_t off = base + j * inner;
            dot += go[off] * y[off];
        }
        for (size_t j = 0; j < reduce; ++j) {
            const size_t off = base + j * inner;
            gi[off] = y[off] * (go[off] - dot);
        }
    }
}

// ---- rows (inner == 1) ---------------------------------------------------------
//
// A workgroup of W waves takes RW rows; wave w holds columns [64 w CPL, 64
// (w + 1) CPL) of each, lane l column 64 i + l of them in register i.  HBM is
// the floor (8 B per element forward, 12 B backward: the elements are read
// once and stay in registers); the sum is a chain of one dependent fp32
// addition per column, so a wave adds its RW rows side by side, a lane each:
// the values pass through LDS 256 columns at a time, and a lane reads its row
// four columns to a read, the reads of the next 16 columns issued before the
// additions of the last.  The waves of a workgroup take their turns in column
// order (W - 1 barriers).  The columns past the row are +0 terms: both sums
// start from +0 and are never -0, so a +0 changes nothing.
//
// s (lane r < RW: row r's running sum) plus STEP columns of row p in order.
template <int STEP>
__device__ __forceinline__ float row_chain(const float *p, float s) {
    static_assert(STEP % 32 == 0, "two halves of 16 columns");
    float4 q[2][4];
    auto read = [&](float4(&d)[4], int j) {
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = *reinterpret_cast<const float4 *>(p + j + 4 * k);
    };
    auto add = [&](const float4(&d)[4]) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            s += d[k].x;
            s += d[k].y;
            s += d[k].z;
            s += d[k].w;
        }
    };
    read(q[0], 0);
#pragma unroll 1
    for (int j = 0; j < STEP; j += 32) {
        read(q[1], j + 16);
        __builtin_amdgcn_sched_barrier(0);  // the reads before the additions they overlap
        add(q[0]);
        read(q[0], j + 32 < STEP ? j + 32 : j);
        __builtin_amdgcn_sched_barrier(0);
        add(q[1]);
    }
    return s;
}

// The sum over the columns, in order, of term(r, i) (0 past the row), for every
// row r of the workgroup, returned to all its threads.
template <int RW, int CPL, int W, class Term>
__device__ __forceinline__ void row_sums(Term term, int cols, int lane, int wave, float (&sum)[RW]) {
    constexpr int S = CPL < 4 ? CPL : 4;  // registers per step
    static_assert(CPL % S == 0, "whole steps");
    // rows start 4 banks apart; one tile, the waves' turns are a barrier apart
    __shared__ __attribute__((aligned(16))) float tile[RW][64 * S + 4];
    __shared__ float carry[RW];
    float s = 0.0f;
#pragma unroll 1
    for (int w = 0; w < W; ++w) {
        if (w == wave) {  // uniform
            if (w > 0) s = carry[lane < RW ? lane : 0];
#pragma unroll
            for (int i0 = 0; i0 < CPL; i0 += S) {
                if (64 * (wave * CPL + i0) >= cols) break;  // uniform: past the row
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int i = 0; i < S; ++i) tile[r][64 * i + lane] = term(r, i0 + i);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                s = row_chain<64 * S>(tile[lane < RW ? lane : 0], s);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            if (W > 1 && lane < RW) carry[lane] = s;
        }
        if (W > 1) __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) sum[r] = W > 1 ? carry[r] : __shfl(s, r, 64);
}

template <int RW, int CPL, int W>
__global__ __launch_bounds__(64 * W) void softmax_rows_fwd(const float *__restrict__ x, float *__restrict__ y,
                                                           size_t rows, int cols) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t row0 = static_cast<size_t>(blockIdx.x) * RW;
    const int c0 = wave * 64 * CPL + lane;
    float e[RW][CPL], m[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const float *p = x + (row0 + r < rows ? row0 + r : rows - 1) * cols;
#pragma unroll
        for (int i = 0; i < CPL; ++i) e[r][i] = p[min(c0 + 64 * i, cols - 1)];
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {  // a clamped load repeats the row's last element: the same maximum
        float v = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < CPL; ++i) v = fmaxf(v, e[r][i]);
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
        m[r] = v;
    }
    if constexpr (W > 1) {
        __shared__ float wm[W][RW];
        if (lane == 0)
#pragma unroll
            for (int r = 0; r < RW; ++r) wm[wave][r] = m[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int w = 0; w < W; ++w) m[r] = fmaxf(m[r], wm[w][r]);
    }
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int i = 0; i < CPL; ++i) e[r][i] = c0 + 64 * i < cols ? softmax_exp(e[r][i] - m[r]) : 0.0f;
    float sum[RW];
    row_sums<RW, CPL, W>([&](int r, int i) { return e[r][i]; }, cols, lane, wave, sum);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const float inv = 1.0f / sum[r];
        if (row0 + r < rows) {  // uniform
            float *q = y + (row0 + r) * cols;
#pragma unroll
            for (int i = 0; i < CPL; ++i)
                if (c0 + 64 * i < cols) q[c0 + 64 * i] = e[r][i] * inv;
        }
    }
}

template <int RW, int CPL, int W>
__global__ __launch_bounds__(64 * W) void softmax_rows_bwd(const float *__restrict__ y, const float *__restrict__ go,
                                                           float *__restrict__ gi, size_t rows, int cols) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t row0 = static_cast<size_t>(blockIdx.x) * RW;
    const int c0 = wave * 64 * CPL + lane;
    float yv[RW][CPL], gv[RW][CPL];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const size_t at = (row0 + r < rows ? row0 + r : rows - 1) * cols;
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            const int c = min(c0 + 64 * i, cols - 1);
            yv[r][i] = y[at + c];
            gv[r][i] = go[at + c];
        }
    }
    float dot[RW];
    row_sums<RW, CPL, W>([&](int r, int i) { return c0 + 64 * i < cols ? gv[r][i] * yv[r][i] : 0.0f; }, cols, lane,
                         wave, dot);
#pragma unroll
    for (int r = 0; r < RW; ++r)
        if (row0 + r < rows) {  // uniform
            float *q = gi + (row0 + r) * cols;
#pragma unroll
            for (int i = 0; i < CPL; ++i)
                if (c0 + 64 * i < cols) q[c0 + 64 * i] = yv[r][i] * (gv[r][i] - dot[r]);
        }
}

// ---- long rows (inner == 1) ----------------------------------------------------
//
// Past a few thousand columns a row's registers leave room for 2 to 4 rows a
// CU, and the chain of additions (4 ns a column) is all that runs.  Here a
// workgroup takes 8 rows without holding them: four waves, two rows each, read
// 256 columns ahead and leave their terms in LDS, a fifth adds the eight rows
// side by side, one chunk behind (a barrier a chunk, two tiles).  The columns
// are read again for the maximum and for the results (exp taken twice: the
// same bits).
constexpr int kLongRows = 8, kLongOwn = 2, kLongChunk = 256, kLongBlock = 64 * (1 + kLongRows / kLongOwn);

// sum[i]: the sum over the columns, in order, of term(v, i, c) of the wave's
// row i, v = load(i, c) for c in range.
template <class Load, class Term>
__device__ __forceinline__ void long_sums(Load load, Term term, int cols, int lane, int wave, float (&sum)[kLongOwn]) {
    constexpr int S = kLongChunk / 64;
    // rows start 4 banks apart
    __shared__ __attribute__((aligned(16))) float tile[2][kLongRows][kLongChunk + 4];
    __shared__ float total[kLongRows];
    const int chunks = (cols + kLongChunk - 1) / kLongChunk;
    const int own = wave > 0 ? (wave - 1) * kLongOwn : 0;
    using V = decltype(load(0, 0));
    V v[kLongOwn][S], next[kLongOwn][S];
    auto fetch = [&](V(&d)[kLongOwn][S], int k) {
#pragma unroll
        for (int i = 0; i < kLongOwn; ++i)
#pragma unroll
            for (int j = 0; j < S; ++j) d[i][j] = load(i, min(k * kLongChunk + 64 * j + lane, cols - 1));
    };
    if (wave > 0) fetch(v, 0);
    float s = 0.0f;
#pragma unroll 1
    for (int k = 0; k <= chunks; ++k) {
        if (wave > 0) {  // uniform
            if (k < chunks) {
                fetch(next, min(k + 1, chunks - 1));
#pragma unroll
                for (int i = 0; i < kLongOwn; ++i)
#pragma unroll
                    for (int j = 0; j < S; ++j) {
                        const int c = k * kLongChunk + 64 * j + lane;
                        tile[k & 1][own + i][64 * j + lane] = c < cols ? term(v[i][j], i) : 0.0f;
                        v[i][j] = next[i][j];
                    }
            }
        } else if (k > 0) {
            s = row_chain<kLongChunk>(tile[(k - 1) & 1][lane < kLongRows ? lane : 0], s);
        }
        __syncthreads();
    }
    if (wave == 0 && lane < kLongRows) total[lane] = s;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kLongOwn; ++i) sum[i] = total[own + i];
}

__global__ __launch_bounds__(kLongBlock) void softmax_long_fwd(const float *__restrict__ x, float *__restrict__ y,
                                                               size_t rows, int cols) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t first = static_cast<size_t>(blockIdx.x) * kLongRows + (wave > 0 ? (wave - 1) * kLongOwn : 0);
    const float *p[kLongOwn];
    float m[kLongOwn], sum[kLongOwn];
#pragma unroll
    for (int i = 0; i < kLongOwn; ++i) {
        p[i] = x + min(first + i, rows - 1) * cols;
        m[i] = -__builtin_inff();
    }
    if (wave > 0) {
        for (int c = lane; c < cols; c += 64 * 16) {
            float v[kLongOwn][16];  // a clamped load repeats the row's last element: the same maximum
#pragma unroll
            for (int i = 0; i < kLongOwn; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) v[i][j] = p[i][min(c + 64 * j, cols - 1)];
#pragma unroll
            for (int i = 0; i < kLongOwn; ++i)
#pragma unroll
                for (int j = 0; j < 16; ++j) m[i] = fmaxf(m[i], v[i][j]);
        }
#pragma unroll
        for (int i = 0; i < kLongOwn; ++i)
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) m[i] = fmaxf(m[i], __shfl_xor(m[i], d, 64));
    }
    long_sums([&](int i, int c) { return p[i][c]; }, [&](float v, int i) { return softmax_exp(v - m[i]); }, cols, lane,
              wave, sum);
    if (wave == 0) return;
#pragma unroll
    for (int i = 0; i < kLongOwn; ++i) {
        if (first + i >= rows) break;  // uniform
        const float inv = 1.0f / sum[i];
        float *q = y + (first + i) * cols;
        for (int c = lane; c < cols; c += 64 * 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = p[i][min(c + 64 * j, cols - 1)];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (c + 64 * j < cols) q[c + 64 * j] = softmax_exp(v[j] - m[i]) * inv;
        }
    }
}

__global__ __launch_bounds__(kLongBlock) void softmax_long_bwd(const float *__restrict__ y,
                                                               const float *__restrict__ go, float *__restrict__ gi,
                                                               size_t rows, int cols) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t first = static_cast<size_t>(blockIdx.x) * kLongRows + (wave > 0 ? (wave - 1) * kLongOwn : 0);
    size_t at[kLongOwn];
    float dot[kLongOwn];
#pragma unroll
    for (int i = 0; i < kLongOwn; ++i) at[i] = min(first + i, rows - 1) * cols;
    long_sums([&](int i, int c) { return make_float2(y[at[i] + c], go[at[i] + c]); },
              [&](float2 v, int) { return v.y * v.x; }, cols, lane, wave, dot);
    if (wave == 0) return;
#pragma unroll
    for (int i = 0; i < kLongOwn; ++i) {
        if (first + i >= rows) break;  // uniform
        for (int c = lane; c < cols; c += 64 * 8) {
            float yv[8], gv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const size_t k = at[i] + min(c + 64 * j, cols - 1);
                yv[j] = y[k];
                gv[j] = go[k];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (c + 64 * j < cols) gi[at[i] + c + 64 * j] = yv[j] * (gv[j] - dot[i]);
        }
    }
}

// Rows of this many columns take the row kernels.  From 10 columns on they are
// the faster (2^20 x 10: 123 / 49 us forward / backward against 131 / 111 with
// a thread per row; x 16: 123 / 49 against 424 / 485); past kRegMaxCols a
// workgroup's registers end.
constexpr size_t kRowsMinCols = 10, kRegMaxCols = 32768, kRowsMaxCols = size_t(1) << 30;

// In as many launches as the rows take: a grid holds fewer than 2^32 threads
// (2^29 rows of 10 columns are that many).
template <bool FWD, int RW, int CPL, int W>
static void launch_rows_as(const float *a, const float *b, float *out, size_t rows, int cols, hipStream_t s) {
    constexpr size_t kRows = ((size_t(1) << 32) - 1) / (64 * W) * RW;
    for (size_t r = 0; r < rows; r += kRows) {
        const size_t n = rows - r < kRows ? rows - r : kRows, at = r * cols;
        const dim3 grid(static_cast<unsigned>((n + RW - 1) / RW)), block(64 * W);
        if constexpr (FWD) launch((softmax_rows_fwd<RW, CPL, W>), grid, block, 0, s, a + at, out + at, n, cols);
        else launch((softmax_rows_bwd<RW, CPL, W>), grid, block, 0, s, a + at, b + at, out + at, n, cols);
    }
}

// Past 4096 columns a CU's registers hold 4 rows, 2 or 1, and a round of them
// takes a chain of additions; the long kernels' workgroups are slower one by
// one (their reads are waited for, 3 us a chunk), but more of them run at once.
// The line is at 3.5 rounds.  us forward / backward, registers then long: 8192 x
// 8000 380 / 361, 303 / 260; 4096 x 12320 484 / 449, 265 / 220; 1804 x 12320
// 239 / 224, 188 / 124; 1000 x 25000 432 / 501, 368 / 241; below it 1024 x 8000
// 50 / 48, 119 / 78; 512 x 12320 62 / 58, 168 / 116.  Past kRegMaxCols there are
// only these and a thread per row (64 x 100000: 1290 / 899, a thread per row 64600 / 36100).
static bool rows_are_long(size_t rows, size_t cols) {
    if (cols <= 4096) return false;
    const size_t held = cols <= 8192 ? 4 : cols <= 16384 ? 2 : 1;
    return cols > kRegMaxCols || 2 * rows > 7 * held * static_cast<size_t>(device_cu_count());
}

// More rows side by side while a row is short (their chains share the adds'
// issue slots), then as many waves as the row needs at 8 columns a lane, the
// rows of a workgroup halved and the columns of a lane doubled for the last.
// (The backward forms of 16 waves have 128 registers a lane for two operands
// and spill 10, 8 and 20 of them.)  From 2049 columns on the waves that wait for their turn show: where the rows
// fill the chip, half as many at 16 columns a lane (us forward / backward, 16384 x
// 4000: 247 / 342 with eight, 199 / 210 with four; 2048 x 4000: 33 / 47 and 37 / 30;
// 512 x 4000: 26 / 20 and 31 / 21).
template <bool FWD>
static bool launch_rows(const float *a, const float *b, float *out, size_t rows, size_t cols, hipStream_t s) {
    if (cols < kRowsMinCols || cols > kRowsMaxCols || rows > 0x7fffffffULL) return false;
    if (rows_are_long(rows, cols)) {
        const dim3 grid(static_cast<unsigned>((rows + kLongRows - 1) / kLongRows)), block(kLongBlock);
        if constexpr (FWD) launch(softmax_long_fwd, grid, block, 0, s, a, out, rows, static_cast<int>(cols));
        else launch(softmax_long_bwd, grid, block, 0, s, a, b, out, rows, static_cast<int>(cols));
        return true;
    }
    const bool four = rows > (FWD ? 8 : 4) * static_cast<size_t>(device_cu_count());
    const int c = static_cast<int>(cols);
    if (c <= 64) launch_rows_as<FWD, 8, 1, 1>(a, b, out, rows, c, s);
    else if (c <= 128) launch_rows_as<FWD, 8, 2, 1>(a, b, out, rows, c, s);
    else if (c <= 256) launch_rows_as<FWD, 8, 4, 1>(a, b, out, rows, c, s);
    else if (c <= 512) launch_rows_as<FWD, 4, 8, 1>(a, b, out, rows, c, s);
    else if (c <= 1024) launch_rows_as<FWD, 4, 8, 2>(a, b, out, rows, c, s);
    else if (c <= 2048) launch_rows_as<FWD, 4, 8, 4>(a, b, out, rows, c, s);
    else if (c <= 4096 && four) launch_rows_as<FWD, 4, 16, 4>(a, b, out, rows, c, s);
    else if (c <= 4096) launch_rows_as<FWD, 4, 8, 8>(a, b, out, rows, c, s);
    else if (c <= 8192) launch_rows_as<FWD, 4, 8, 16>(a, b, out, rows, c, s);
    else if (c <= 16384) launch_rows_as<FWD, 2, 16, 16>(a, b, out, rows, c, s);
    else launch_rows_as<FWD, 1, 32, 16>(a, b, out, rows, c, s);
    return true;
}

}  // namespace tship

using namespace tship;

extern "C" {

int ts_hip_softmax(const float *x, float *y, size_t outer, size_t reduce, size_t inner, void *stream) {
    const size_t slices = outer * inner;
    if (slices == 0 || reduce == 0) return reduce == 0 && slices ? TS_HIP_EINVAL : TS_HIP_OK;
    if (!x || !y) return TS_HIP_EINVAL;
    if (inner == 1 && launch_rows<true>(x, nullptr, y, outer, reduce, as_stream(stream))) return launch_status();
    launch(softmax_fwd, dim3(grid_for(slices)), dim3(kBlock), 0, as_stream(stream), x, y, outer,
                       reduce, inner);
    return launch_status();
}

int ts_hip_softmax_backward(const float *y, const float *go, float *gi, size_t outer, size_t reduce,
                            size_t inner, void *stream) {
    const size_t slices = outer * inner;
    if (slices == 0 || reduce == 0) return TS_HIP_OK;
    if (!y || !go || !gi) return TS_HIP_EINVAL;
    if (inner == 1 && launch_rows<false>(y, go, gi, outer, reduce, as_stream(stream))) return launch_status();
    launch(softmax_bwd, dim3(grid_for(slices)), dim3(kBlock), 0, as_stream(stream), y, go, gi,
                       outer, reduce, inner);
    return launch_status();
}

}  // extern "C"
