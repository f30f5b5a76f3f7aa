// Shape-general kernels: NumPy broadcasting (tensor/ops/broadcasting.rs:
// 299-478) and sums over any set of axes (sum_dims / mean_dims,
// tensor/reductions/{sum,mean}.rs, and the gradient reduction of
// grad_fn/utils.rs:23-60), up to rank 8.
//
// broadcast_gather: out[i] = src[offset of i's coordinates], with the source
// strides of broadcast axes set to 0 -- the reference materialises the same
// values with broadcast_copy_data.  HBM-bound: 4 B written per element, the
// source read through the caches.  Neighbouring axes that are both repeated, or
// both copied, are merged first ([8192, 1] over [8192, 1024] is two axes, a bias
// over any batch two); below 2^31 elements a thread then writes four
// consecutive ones (broadcast_quads) and finds their coordinates with
// multiplications: a 64-bit division per element and axis had bound the copy
// (8192 x 1024: 24 us, now 8).
//
// reduce_axes: output element o (keepdim layout) sums the input elements
// whose kept coordinates equal o's, in f64, in a fixed order: G lanes per
// output (1, 64 or 256, chosen from the shape) each add a strided share of
// the reduced index space, then a shuffle / LDS tree combines them.
#include "ts_hip_internal.h"

namespace tship {

constexpr int kMaxRank = 8;

struct Layout {
    int rank;
    uint64_t dims[kMaxRank];
    uint64_t src_stride[kMaxRank];  // element stride in the source per output axis
};

__global__ __launch_bounds__(kBlock) void broadcast_gather(const float *__restrict__ src,
                                                           float *__restrict__ out, size_t n,
                                                           Layout L, float scale, int use_scale) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        size_t rem = i, off = 0;
        for (int k = L.rank - 1; k >= 0; --k) {
            const uint64_t c = rem % L.dims[k];
            rem /= L.dims[k];
            off += c * L.src_stride[k];
        }
        const float v = src[off];
        out[i] = use_scale ? v * scale : v;
    }
}

// x / d for x < 2^31: the quotient's multiplier is 2^32 (2^l - d) / d + 1 with
// 2^l the power of two at or above d (Granlund and Montgomery, "Division by
// invariant integers using multiplication").
struct FastDiv {
    uint32_t d, m, l;
};
static FastDiv fast_div(uint32_t d) {
    FastDiv f{d, 0, 0};
    while (f.l < 31 && (uint32_t(1) << f.l) < d) ++f.l;
    f.m = static_cast<uint32_t>(((uint64_t(1) << 32) * ((uint64_t(1) << f.l) - d)) / d + 1);
    return f;
}
__device__ __forceinline__ uint32_t quotient(uint32_t x, const FastDiv &f) { return (__umulhi(x, f.m) + x) >> f.l; }

struct QuadLayout {
    int rank;                    // merged axes, innermost first
    FastDiv dim[kMaxRank];
    uint32_t stride[kMaxRank];   // in the source; 0 repeated
};

__device__ __forceinline__ uint32_t quad_offset(const QuadLayout &L, uint32_t i) {
    uint32_t off = 0;
#pragma unroll
    for (int k = 0; k < kMaxRank; ++k) {
        if (k < L.rank - 1) {
            const uint32_t q = quotient(i, L.dim[k]);
            off += (i - q * L.dim[k].d) * L.stride[k];
            i = q;
        }
    }
    return off + i * L.stride[L.rank - 1];
}

// INNER: the innermost axis is a multiple of four long, so a thread's four
// elements share the outer coordinates.  VEC: out is 16-byte aligned.
template <bool INNER, bool VEC>
__global__ __launch_bounds__(kBlock) void broadcast_quads(const float *__restrict__ src, float *__restrict__ out,
                                                          uint32_t n, QuadLayout L, float scale, int use_scale) {
    const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) * 4;
    if (i >= n) return;
    f4v_t v;
    if (INNER) {
        const uint32_t off = quad_offset(L, i), s = L.stride[0];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = src[off + c * s];
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = src[quad_offset(L, min(i + c, n - 1))];
    }
    if (use_scale) {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = v[c] * scale;
    }
    if (VEC && i + 3 < n) {
        *reinterpret_cast<f4v_t *>(out + i) = v;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (i + c < n) out[i + c] = v[c];
    }
}

// Two operands broadcast against each other (broadcast_binary): the same groups
// of four and merged axes, with a stride per operand, so neither is written out
// in full first.
struct PairLayout {
    int rank;  // merged axes, innermost first
    FastDiv dim[kMaxRank];
    uint32_t sa[kMaxRank], sb[kMaxRank];
};
__device__ __forceinline__ void pair_offsets(const PairLayout &L, uint32_t i, uint32_t &oa, uint32_t &ob) {
    oa = ob = 0;
#pragma unroll
    for (int k = 0; k < kMaxRank; ++k) {
        if (k < L.rank - 1) {
            const uint32_t q = quotient(i, L.dim[k]), r = i - q * L.dim[k].d;
            oa += r * L.sa[k];
            ob += r * L.sb[k];
            i = q;
        }
    }
    oa += i * L.sa[L.rank - 1];
    ob += i * L.sb[L.rank - 1];
}

typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

// OP: 0 add, 1 sub, 2 mul, 3 div (its zero divisors from check_start on as
// ts_hip_div reports them).  INNER: the innermost axis is a multiple of four
// long (each operand is read along it by fours, or repeats one value).
// HBM-bound: 8192 x 1024 divided by a column 14 us, where the column written
// out in full and the division after it took 26.
template <int OP, bool INNER>
__global__ __launch_bounds__(kBlock) void broadcast_binary(const float *__restrict__ a, const float *__restrict__ b,
                                                           float *__restrict__ out, uint32_t n, PairLayout L, int vec,
                                                           uint32_t check_start, unsigned long long *zero_index) {
    const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) * 4;
    if (i >= n) return;
    f4v_t x, y, v;
    if (INNER) {
        uint32_t oa, ob;
        pair_offsets(L, i, oa, ob);
        if (L.sa[0]) x = *reinterpret_cast<const f4u_t *>(a + oa);
        else x = f4v_t{a[oa], a[oa], a[oa], a[oa]};
        if (L.sb[0]) y = *reinterpret_cast<const f4u_t *>(b + ob);
        else y = f4v_t{b[ob], b[ob], b[ob], b[ob]};
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t oa, ob;
            pair_offsets(L, min(i + c, n - 1), oa, ob);
            x[c] = a[oa];
            y[c] = b[ob];
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        v[c] = OP == 0 ? x[c] + y[c] : OP == 1 ? x[c] - y[c] : OP == 2 ? x[c] * y[c] : x[c] / y[c];
        if (OP == 3 && zero_index && y[c] == 0.0f && i + c >= check_start && i + c < n)
            atomicMin(zero_index, (unsigned long long)(i + c));
    }
    if (vec && i + 3 < n) {
        *reinterpret_cast<f4v_t *>(out + i) = v;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (i + c < n) out[i + c] = v[c];
    }
}

struct Reduction {
    int kept_rank, red_rank;
    uint64_t kept_dims[kMaxRank], kept_stride[kMaxRank];  // input strides of the kept axes
    uint64_t red_dims[kMaxRank], red_stride[kMaxRank];    // input strides of the reduced axes
    uint64_t n_out, n_red;
};

__device__ inline uint64_t kept_offset(const Reduction &R, uint64_t o) {
    uint64_t off = 0;
    for (int k = R.kept_rank - 1; k >= 0; --k) {
        off += (o % R.kept_dims[k]) * R.kept_stride[k];
        o /= R.kept_dims[k];
    }
    return off;
}

__device__ inline uint64_t red_offset(const Reduction &R, uint64_t r) {
    uint64_t off = 0;
    for (int k = R.red_rank - 1; k >= 0; --k) {
        off += (r % R.red_dims[k]) * R.red_stride[k];
        r /= R.red_dims[k];
    }
    return off;
}

// G lanes per output; G = 1 (a thread per output), 64 (a wave) or 256 (a workgroup)
template <int G>
__global__ __launch_bounds__(kBlock) void reduce_axes(const float *__restrict__ x, float *__restrict__ out,
                                                      Reduction R, float scale, int use_scale) {
    constexpr int kPerBlock = kBlock / G;
    const uint64_t o = static_cast<uint64_t>(blockIdx.x) * kPerBlock + threadIdx.x / G;
    const int lane = threadIdx.x % G;
    double acc = 0.0;
    if (o < R.n_out) {
        const float *p = x + kept_offset(R, o);
        if (R.red_rank == 1) {  // uniform: the reduced axes are one (merged)
            const uint64_t step = G * R.red_stride[0];
            p += lane * R.red_stride[0];
            uint64_t r = lane;
            // eight loads in flight, added in order
            for (; r + 7 * G < R.n_red; r += 8 * G, p += 8 * step) {
                float v[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = p[k * step];
#pragma unroll
                for (int k = 0; k < 8; ++k) acc += static_cast<double>(v[k]);
            }
            for (; r < R.n_red; r += G, p += step) acc += static_cast<double>(*p);
        } else {
            for (uint64_t r = lane; r < R.n_red; r += G) acc += static_cast<double>(p[red_offset(R, r)]);
        }
    }
    if (G >= 64) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d, 64);
    }
    if (G == 256) {
        __shared__ double part[kBlock / 64];
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) acc = ((part[0] + part[1]) + part[2]) + part[3];
    }
    if (lane == 0 && o < R.n_out) {
        const float s = static_cast<float>(acc);
        out[o] = use_scale ? s * scale : s;
    }
}

// ---- transposing two axes (transform/transpose.rs:156-208, materialised) ----
//
// out = src with axes d0 < d1 swapped, both row-major.  Viewing the source as
// [P, D0, M, D1, Q], the output is [P, D1, M, D0, Q].
//
// Q == 1 (d1 is the last axis, as in a matrix transpose): each (p, m) plane
// moves in 64 x 64 tiles through LDS, so a wave reads 64 consecutive floats
// of a source row and writes 64 consecutive floats of an output row; the LDS
// row pitch of 65 floats keeps the column reads conflict-free.  HBM-bound:
// 8 B per element.  Q > 1: runs of Q contiguous floats keep their order, a
// thread per element, reads and writes both along q.

struct TransposeDims {
    uint64_t P, D0, M, D1, Q;
    uint64_t tiles0, tiles1;  // 64-wide tiles along D0 and D1
};

__global__ __launch_bounds__(256) void transpose_tiles(const float *__restrict__ src, float *__restrict__ out,
                                                       TransposeDims T) {
    __shared__ float tile[64][65];
    const uint64_t per_plane = T.tiles0 * T.tiles1;
    const uint64_t b = blockIdx.x;
    const uint64_t plane = b / per_plane, t = b - plane * per_plane;
    const uint64_t i0 = (t / T.tiles1) * 64, j0 = (t % T.tiles1) * 64;
    const uint64_t p = plane / T.M, m = plane - p * T.M;
    const int c = static_cast<int>(threadIdx.x & 63u), r = static_cast<int>(threadIdx.x >> 6);
    // src[p, i, m, j] at ((p * D0 + i) * M + m) * D1 + j
    const float *sb = src + (p * T.D0 * T.M + m) * T.D1;
    const uint64_t in_row = T.M * T.D1;
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint64_t i = i0 + r + 4 * k, j = j0 + c;
        v[k] = (i < T.D0 && j < T.D1) ? sb[i * in_row + j] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) tile[r + 4 * k][c] = v[k];
    __syncthreads();
    // out[p, j, m, i] at ((p * D1 + j) * M + m) * D0 + i
    float *ob = out + (p * T.D1 * T.M + m) * T.D0;
    const uint64_t out_row = T.M * T.D0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint64_t j = j0 + r + 4 * k, i = i0 + c;
        if (i < T.D0 && j < T.D1) ob[j * out_row + i] = tile[c][r + 4 * k];
    }
}

__global__ __launch_bounds__(kBlock) void transpose_runs(const float *__restrict__ src, float *__restrict__ out,
                                                         TransposeDims T, uint64_t n) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t o = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; o < n; o += stride) {
        uint64_t rest = o / T.Q;
        const uint64_t q = o - rest * T.Q;
        const uint64_t i = rest % T.D0;
        rest /= T.D0;
        const uint64_t m = rest % T.M;
        rest /= T.M;
        const uint64_t j = rest % T.D1, p = rest / T.D1;
        out[o] = src[(((p * T.D0 + i) * T.M + m) * T.D1 + j) * T.Q + q];
    }
}

}  // namespace tship

using namespace tship;

extern "C" {

int ts_hip_transpose(const float *src, const size_t *dims, size_t rank, size_t d0, size_t d1, float *out,
                     void *stream) {
    if (rank > 0 && !dims) return TS_HIP_EINVAL;
    if (d0 >= rank || d1 >= rank) return TS_HIP_EINVAL;
    uint64_t n = 1;
    for (size_t k = 0; k < rank; ++k) n *= dims[k];
    if (n == 0) return TS_HIP_OK;
    if (!src || !out) return TS_HIP_EINVAL;
    if (d0 == d1) return ts_hip_copy(src, out, n, stream);
    if (d0 > d1) {
        const size_t t = d0;
        d0 = d1;
        d1 = t;
    }
    TransposeDims T{1, dims[d0], 1, dims[d1], 1, 0, 0};
    for (size_t k = 0; k < d0; ++k) T.P *= dims[k];
    for (size_t k = d0 + 1; k < d1; ++k) T.M *= dims[k];
    for (size_t k = d1 + 1; k < rank; ++k) T.Q *= dims[k];
    hipStream_t s = as_stream(stream);
    if (T.Q == 1) {
        T.tiles0 = (T.D0 + 63) / 64;
        T.tiles1 = (T.D1 + 63) / 64;
        const uint64_t blocks = T.P * T.M * T.tiles0 * T.tiles1;
        if (blocks > 0x7fffffffULL) return TS_HIP_EINVAL;
        launch(transpose_tiles, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, src, out, T);
    } else {
        launch(transpose_runs, dim3(grid_for(n)), dim3(kBlock), 0, s, src, out, T, n);
    }
    return launch_status();
}


int ts_hip_broadcast_copy(const float *src, const size_t *src_dims, size_t src_rank, float *out,
                          const size_t *out_dims, size_t out_rank, float scale, int use_scale,
                          void *stream) {
    if (out_rank > static_cast<size_t>(kMaxRank) || src_rank > out_rank) return TS_HIP_EINVAL;
    if ((src_rank && !src_dims) || (out_rank && !out_dims)) return TS_HIP_EINVAL;
    size_t n = 1;
    for (size_t k = 0; k < out_rank; ++k) n *= out_dims[k];
    if (n == 0) return TS_HIP_OK;
    if (!src || !out) return TS_HIP_EINVAL;
    Layout L{};
    L.rank = static_cast<int>(out_rank);
    // source axes align to the right; a source axis of size 1 (or a missing one) repeats
    size_t stride = 1;
    for (size_t k = out_rank; k-- > 0;) {
        L.dims[k] = out_dims[k];
        const size_t j = k + src_rank - out_rank;  // wraps when the source lacks the axis
        if (k + src_rank >= out_rank) {
            const size_t d = src_dims[j];
            if (d != out_dims[k] && d != 1) return TS_HIP_EINVAL;
            L.src_stride[k] = (d == 1) ? 0 : stride;
            stride *= d;
        } else {
            L.src_stride[k] = 0;
        }
    }
    if (L.rank == 0) {  // scalar to scalar
        L.rank = 1;
        L.dims[0] = 1;
        L.src_stride[0] = 0;
    }
    if (n < (size_t(1) << 31)) {
        // merged axes, innermost first; axes of one element take no part
        QuadLayout Q{};
        uint64_t len[kMaxRank], str[kMaxRank];
        for (int k = L.rank - 1; k >= 0; --k) {
            if (L.dims[k] == 1) continue;
            const int t = Q.rank - 1;
            if (Q.rank && (str[t] == 0 ? L.src_stride[k] == 0 : L.src_stride[k] == str[t] * len[t])) {
                len[t] *= L.dims[k];
            } else {
                len[Q.rank] = L.dims[k];
                str[Q.rank++] = L.src_stride[k];
            }
        }
        if (Q.rank == 0) {
            len[0] = 1;
            str[Q.rank++] = 0;
        }
        for (int k = 0; k < Q.rank; ++k) {
            Q.dim[k] = fast_div(static_cast<uint32_t>(len[k]));
            Q.stride[k] = static_cast<uint32_t>(str[k]);
        }
        const bool inner = len[0] % 4 == 0, vec = aligned16(out);
        const dim3 grid(static_cast<unsigned>((n + 4 * kBlock - 1) / (4 * kBlock))), block(kBlock);
        hipStream_t s = as_stream(stream);
        const uint32_t n32 = static_cast<uint32_t>(n);
        if (inner && vec) launch((broadcast_quads<true, true>), grid, block, 0, s, src, out, n32, Q, scale, use_scale);
        else if (inner) launch((broadcast_quads<true, false>), grid, block, 0, s, src, out, n32, Q, scale, use_scale);
        else if (vec) launch((broadcast_quads<false, true>), grid, block, 0, s, src, out, n32, Q, scale, use_scale);
        else launch((broadcast_quads<false, false>), grid, block, 0, s, src, out, n32, Q, scale, use_scale);
        return launch_status();
    }
    launch(broadcast_gather, dim3(grid_for(n)), dim3(kBlock), 0, as_stream(stream), src, out, n, L,
                       scale, use_scale);
    return launch_status();
}

int ts_hip_broadcast_binary(int op, const float *a, const size_t *a_dims, size_t a_rank, const float *b,
                            const size_t *b_dims, size_t b_rank, float *out, const size_t *out_dims, size_t out_rank,
                            size_t zero_check_start, unsigned long long *zero_index, void *stream) {
    if (op < 0 || op > 3 || out_rank > static_cast<size_t>(kMaxRank) || a_rank > out_rank || b_rank > out_rank)
        return TS_HIP_EINVAL;
    if ((a_rank && !a_dims) || (b_rank && !b_dims) || (out_rank && !out_dims)) return TS_HIP_EINVAL;
    size_t n = 1;
    for (size_t k = 0; k < out_rank; ++k) {
        if (out_dims[k] && n > (size_t(1) << 31) / out_dims[k]) return TS_HIP_EINVAL;
        n *= out_dims[k];
    }
    if (n == 0) return TS_HIP_OK;
    if (n >= (size_t(1) << 31) || !a || !b || !out) return TS_HIP_EINVAL;
    PairLayout L{};
    uint64_t len[kMaxRank], sa[kMaxRank], sb[kMaxRank];
    uint64_t full_a = 1, full_b = 1;  // the operands' strides so far
    for (size_t j = 0; j < out_rank; ++j) {  // innermost first
        const uint64_t d = out_dims[out_rank - 1 - j];
        const uint64_t da = j < a_rank ? a_dims[a_rank - 1 - j] : 1, db = j < b_rank ? b_dims[b_rank - 1 - j] : 1;
        if ((da != d && da != 1) || (db != d && db != 1)) return TS_HIP_EINVAL;
        if (d == 1) continue;
        const uint64_t ta = da == 1 ? 0 : full_a, tb = db == 1 ? 0 : full_b;
        full_a *= da;
        full_b *= db;
        const int t = L.rank - 1;
        auto joins = [&](uint64_t last, uint64_t stride) { return last == 0 ? stride == 0 : stride == last * len[t]; };
        if (L.rank && joins(sa[t], ta) && joins(sb[t], tb)) {
            len[t] *= d;
            continue;
        }
        len[L.rank] = d;
        sa[L.rank] = ta;
        sb[L.rank++] = tb;
    }
    if (L.rank == 0) {
        len[0] = 1;
        sa[0] = sb[0] = 0;
        L.rank = 1;
    }
    for (int k = 0; k < L.rank; ++k) {
        L.dim[k] = fast_div(static_cast<uint32_t>(len[k]));
        L.sa[k] = static_cast<uint32_t>(sa[k]);
        L.sb[k] = static_cast<uint32_t>(sb[k]);
    }
    const bool inner = len[0] % 4 == 0;
    const int vec = aligned16(out) ? 1 : 0;
    const uint32_t n32 = static_cast<uint32_t>(n);
    const uint32_t check = zero_check_start > n ? n32 : static_cast<uint32_t>(zero_check_start);
    const dim3 grid(static_cast<unsigned>((n + 4 * kBlock - 1) / (4 * kBlock))), block(kBlock);
    hipStream_t s = as_stream(stream);
    auto go = [&](auto kernel) { launch(kernel, grid, block, 0, s, a, b, out, n32, L, vec, check, zero_index); };
    switch (op) {
        case 0: inner ? go(broadcast_binary<0, true>) : go(broadcast_binary<0, false>); break;
        case 1: inner ? go(broadcast_binary<1, true>) : go(broadcast_binary<1, false>); break;
        case 2: inner ? go(broadcast_binary<2, true>) : go(broadcast_binary<2, false>); break;
        default: inner ? go(broadcast_binary<3, true>) : go(broadcast_binary<3, false>); break;
    }
    return launch_status();
}

int ts_hip_reduce_sum(const float *x, const size_t *dims, size_t rank, unsigned reduce_mask, float *out,
                      float scale, int use_scale, void *stream) {
    if (rank > static_cast<size_t>(kMaxRank) || (rank && !dims)) return TS_HIP_EINVAL;
    if (rank < 32 && (reduce_mask >> rank) != 0) return TS_HIP_EINVAL;
    Reduction R{};
    uint64_t stride = 1, n_in = 1;
    uint64_t st[kMaxRank];
    for (size_t k = rank; k-- > 0;) {
        st[k] = stride;
        stride *= dims[k];
    }
    n_in = stride;
    R.n_out = 1;
    R.n_red = 1;
    // neighbouring axes of a kind merged (the same element order), axes of one
    // element left out
    auto axis = [](int &r, uint64_t *d, uint64_t *s, uint64_t len, uint64_t stride, bool joins) {
        if (joins) {
            d[r - 1] *= len;
            s[r - 1] = stride;
        } else {
            d[r] = len;
            s[r++] = stride;
        }
    };
    int last = -1;  // the kind of the last axis taken
    for (size_t k = 0; k < rank; ++k) {
        const int kind = (reduce_mask >> k) & 1u;
        (kind ? R.n_red : R.n_out) *= dims[k];
        if (dims[k] == 1) continue;
        if (kind) axis(R.red_rank, R.red_dims, R.red_stride, dims[k], st[k], last == 1);
        else axis(R.kept_rank, R.kept_dims, R.kept_stride, dims[k], st[k], last == 0);
        last = kind;
    }
    if (R.n_out == 0) return TS_HIP_OK;
    if (!out) return TS_HIP_EINVAL;
    if (n_in == 0) return ts_hip_fill(out, 0.0f, R.n_out, stream);  // empty sums are 0
    if (!x) return TS_HIP_EINVAL;
    if (R.kept_rank == 0) {  // everything reduced: one output
        R.kept_rank = 1;
        R.kept_dims[0] = 1;
        R.kept_stride[0] = 0;
    }
    if (R.red_rank == 0) {
        R.red_rank = 1;
        R.red_dims[0] = 1;
        R.red_stride[0] = 0;
    }
    hipStream_t s = as_stream(stream);
    const uint64_t cus = static_cast<uint64_t>(device_cu_count());
    if (R.n_out >= cus * 256 || R.n_red < 64) {
        const uint64_t blocks = (R.n_out + kBlock - 1) / kBlock;
        if (blocks > 0x7fffffffULL) return TS_HIP_EINVAL;
        launch(reduce_axes<1>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s, x, out, R,
                           scale, use_scale);
    } else if (R.n_out >= cus * 4) {
        const uint64_t blocks = (R.n_out + 3) / 4;
        launch(reduce_axes<64>, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s, x, out, R,
                           scale, use_scale);
    } else {
        launch(reduce_axes<256>, dim3(static_cast<unsigned>(R.n_out)), dim3(kBlock), 0, s, x, out,
                           R, scale, use_scale);
    }
    return launch_status();
}

}  // extern "C"
