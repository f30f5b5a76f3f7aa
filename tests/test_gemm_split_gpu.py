"""Products on the bf16 matrix cores (2.2e9 operations and more, 1.5e9 of ragged sizes): every layout at
the edges of the tiles and of the stages of k, odd leading dimensions and addresses, operands of any range,
the tiles that are left to the fp32 instructions, and one result from every entry point.

Bound, per element, in units of 2^-24 of sum |a| |b|: the pieces' products left out are below 1; six
instructions add a stage of 16 k from zero, each dropping less than 2 of that stage's sum |a| |b|: 12 in all;
a stage joins the running sum, and the four groups' sums each other, with one rounding: K / 16 + 2 + 4; and
the result takes one more when its scale is taken back (to the subnormal grid where it is that small).
The fp32 instructions' bound, one rounding a term, is K: the larger for K >= 64."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_bits_equal, normal

pytestmark = pytest.mark.gpu


def _bound(K, mag):
    return (20 + K / 16) * 2.0 ** -24 * mag + 2.0 ** -149


# (trans_a, trans_b, M, N, K, operand pitch pad, operand offset in floats)
CASES = [
    (0, 0, 4224, 4224, 256, 0, 0),      # 128x128 tiles, two a CU
    (0, 1, 4096, 4096, 256, 0, 0),
    (1, 0, 4096, 4096, 256, 0, 0),
    (1, 1, 4096, 4096, 256, 0, 0),
    (0, 0, 4090, 4093, 225, 0, 1),      # ragged, a partial stage of one k, no aligned address
    (0, 1, 4095, 4091, 255, 3, 1),
    (1, 0, 4093, 4094, 224, 0, 1),
    (1, 1, 4089, 4090, 193, 1, 3),
    (0, 0, 2048, 1408, 640, 0, 0),      # 128x128 tiles, two groups
    (0, 1, 2049, 1409, 641, 0, 0),
    (1, 0, 2051, 1411, 643, 1, 0),
    (1, 1, 2050, 1410, 642, 0, 1),
    (0, 0, 2049, 4097, 200, 0, 0),      # one group
    (0, 1, 2050, 4099, 191, 1, 1),
    (1, 0, 2051, 4098, 224, 0, 3),
    (1, 1, 2047, 4095, 231, 0, 0),
    (0, 0, 769, 641, 13001, 0, 0),      # 64x64 tiles, four groups, the last one's stages short
    (0, 1, 771, 643, 16383, 0, 1),
    (1, 0, 897, 513, 16000, 3, 0),
    (1, 1, 641, 770, 20011, 0, 0),
    (0, 0, 100, 8130, 1030, 0, 0),      # one row of 64x128 tiles and a part
    (0, 1, 96, 12000, 1004, 0, 1),
    (1, 0, 1531, 777, 1999, 0, 0),      # 64x128 tiles, two groups, one stage more for the first
    (1, 1, 1999, 777, 1063, 1, 0),
    (0, 1, 4097, 67, 4001, 0, 0),       # fewer columns than the wider tiles have
    (0, 0, 4160, 4160, 64, 0, 0),       # the fewest k
    (0, 1, 5001, 4161, 79, 0, 0),
    (1, 0, 25000, 1000, 67, 0, 0),      # few k
    (0, 0, 1280, 1280, 672, 0, 0),      # the smallest
    (1, 0, 999, 777, 1001, 0, 0),
]


def _operand(rows, cols, pad, off, seed, scale=1.0):
    from gpu_util import Dev

    x = normal((rows, cols), seed, scale)
    buf = np.zeros((rows, cols + pad), np.float32)
    buf[:, :cols] = x
    return x, Dev.of(buf, offset=off), cols + pad


def _sample(a, b, ta, tb, rng, M, N):
    """Rows and columns to check (the edges and some inside), their f64 product and sum |a| |b|."""
    i = np.unique(np.concatenate([np.arange(min(M, 20)), M - 1 - np.arange(min(M, 20)), rng.integers(0, M, 40)]))
    j = np.unique(np.concatenate([np.arange(min(N, 20)), N - 1 - np.arange(min(N, 20)), rng.integers(0, N, 40)]))
    A = (a[:, i].T if ta else a[i]).astype(np.float64)
    B = (b[j].T if tb else b[:, j]).astype(np.float64)
    return i, j, A @ B, np.abs(A) @ np.abs(B)


@pytest.mark.parametrize("ta,tb,M,N,K,pad,off", CASES)
def test_split_products(ta, tb, M, N, K, pad, off):
    from gpu_util import Dev, hip, hip_check, sync

    print(f"[split] ta={ta} tb={tb} {M}x{N}x{K} pad={pad} off={off}", flush=True)
    assert 2 * M * N * K >= (1.5e9 if M % 4 or N % 4 or K % 4 else 2.2e9)
    # gradients' magnitudes on one side: far below f16's range before scaling
    a, da, lda = _operand(*((K, M) if ta else (M, K)), pad, off, 31, 1e-9)
    b, db, ldb = _operand(*((N, K) if tb else (K, N)), pad, off, 32)
    ldc = N + pad
    dc = Dev.of(np.full((M, ldc), np.nan, np.float32), offset=off)
    hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, dc.ptr, ldc, None), "ts_hip_gemm")
    sync()
    out = dc.get((M, ldc))
    got = out[:, :N]
    assert np.all(np.isfinite(got))
    if pad:
        assert np.all(np.isnan(out[:, N:])), "the output pitch's padding was written"
    i, j, want, mag = _sample(a, b, ta, tb, np.random.default_rng(1), M, N)
    err = np.abs(got[np.ix_(i, j)] - want)
    assert np.all(err <= _bound(K, mag))
    # and closer than one rounding in two terms, as the fp32 instructions take them, leaves it
    assert np.sqrt(np.mean(err ** 2)) <= 0.3 * np.sqrt(K / 2) * 2.0 ** -24 * np.sqrt(np.mean(want ** 2)) + 2.0 ** -149


# Values of every range in one row: kind, and what it asks of A (M x K) and B (K x N).
def _ranges(kind, A, B, rng):
    K = A.shape[1]
    sel = np.zeros(K, bool)
    share, e = {"a quarter at 2^-45": (0.25, -45), "a fifth at 2^-41": (0.2, -41), "a tenth at 2^-60": (0.1, -60),
                "an eighth at 2^-120": (0.125, -120)}.get(kind, (0, 0))
    if share:  # a few small columns of A, the only ones that B's rows meet
        sel[rng.choice(K, int(share * K), replace=False)] = True
        return np.where(sel, A * np.float32(2.0) ** e, A), np.where(sel[:, None], B, np.float32(0))
    if kind.startswith("opposite halves"):
        s = np.float32(2.0) ** int(kind.split("^")[1])
        half = np.arange(K) % 2 == 0
        return np.where(half, A * s, A), np.where(half[:, None], B, B * s)
    if kind == "term-balanced":
        s = (np.float32(2.0) ** rng.integers(-60, 61, K)).astype(np.float32)
        return A * s, B / s[:, None]
    if kind == "rows of mixed magnitude":
        return A * (np.float32(2.0) ** rng.integers(-40, 41, A.shape)).astype(np.float32), B
    if kind == "both tiny":  # products on the subnormal grid
        return A * np.float32(2.0 ** -66), B * np.float32(2.0 ** -66)
    if kind == "subnormal and huge":
        return (A * np.float32(2.0 ** -126)) * np.float32(2.0 ** -12), B * np.float32(2.0 ** 90)
    if kind == "past the stages' sums":
        return A * np.float32(2.0 ** 70), B * np.float32(2.0 ** 45)
    assert kind == "past the stages' scale"
    return A * np.float32(2.0 ** 115), B * np.float32(2.0 ** -110)


RANGES = ["a quarter at 2^-45", "a fifth at 2^-41", "a tenth at 2^-60", "an eighth at 2^-120", "opposite halves 2^-20",
          "opposite halves 2^-22", "term-balanced", "rows of mixed magnitude", "both tiny", "subnormal and huge",
          "past the stages' scale", "past the stages' sums"]
# one size of each tile: 64x64, 64x128, 128x128 by two groups and by one
TILES = [(769, 770, 1280), (1100, 1300, 1024), (2049, 1409, 643), (3001, 2050, 512)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("kind", RANGES)
def test_split_values_of_any_range(ta, tb, kind):
    from gpu_util import Dev, hip, hip_check, sync

    for M, N, K in TILES:
        print(f"[split, {kind}] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
        rng = np.random.default_rng(K)
        A, B = _ranges(kind, normal((M, K), 41), normal((K, N), 42), rng)
        a, b = (np.ascontiguousarray(A.T) if ta else A), (np.ascontiguousarray(B.T) if tb else B)
        da, db, dc = Dev.of(a), Dev.of(b), Dev(M * N)
        hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, a.shape[1], db.ptr, b.shape[1], dc.ptr, N, None), "gemm")
        sync()
        i, j, want, mag = _sample(a, b, ta, tb, rng, M, N)
        got = dc.get((M, N))[np.ix_(i, j)]
        # (what the fp32 instructions have is within one rounding a term; products below the normal range
        # round to the subnormal grid there)
        tol = K * 2.0 ** -24 * mag + K * 2.0 ** -149 if kind.startswith("past") else _bound(K, mag)
        assert np.all(np.abs(got - want) <= tol), (kind, M, N, K)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split_exact_products(ta, tb):
    # products that are fp32 values come out as they are: by a permutation (values of any magnitude) and of
    # whole numbers; a sum of nothing is +0
    from gpu_util import Dev, hip, hip_check, sync

    for M, N, K in TILES + [(1500, 1024, 1024)]:
        print(f"[split, exact] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
        rng = np.random.default_rng(M)
        A = normal((M, K), 47) * (np.float32(2.0) ** rng.integers(-100, 90, (M, K))).astype(np.float32)
        cols = rng.integers(0, K, N)
        P = np.zeros((K, N), np.float32)
        P[cols, np.arange(N)] = 1
        whole = rng.integers(-4096, 4097, (M, K)).astype(np.float32), rng.integers(-3, 4, (K, N)).astype(np.float32)
        # rows of zeros of either sign, and terms that cancel to nothing
        Z, B = normal((M, K), 48), normal((K, N), 49)
        Z[5], Z[6] = 0.0, -0.0
        Z[7, 1::2] = Z[7, 0:K - K % 2:2]
        Z[7, K - K % 2:] = 0
        B[1:K:2] = -B[0:K - 1:2]
        for X, Y, want, rows in ((A, P, A[:, cols], slice(None)), (*whole, whole[0] @ whole[1], slice(None)),
                                 (Z, B, np.zeros((3, N), np.float32), slice(5, 8))):
            x, y = (np.ascontiguousarray(X.T) if ta else X), (np.ascontiguousarray(Y.T) if tb else Y)
            da, db, dc = Dev.of(x), Dev.of(y), Dev(M * N)
            hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, x.shape[1], db.ptr, y.shape[1], dc.ptr, N, None), "gemm")
            sync()
            assert_bits_equal(dc.get((M, N))[rows], want, f"{M}x{N}x{K}")


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(4224, 4224, 128), (2048, 1409, 640), (1999, 777, 1063), (769, 769, 16001)])
def test_split_tiles_left_to_fp32(ta, tb, M, N, K):
    # op(A)'s rows: 3 an infinity, 130 a NaN, 200 the type's lowest value beside ordinary ones that meet
    # zeros, 257 one outlier of 2^60, 300 tiny values, 301 subnormals, 400 zeros; op(B)'s column 5 an infinity
    from gpu_util import Dev, hip, hip_check, sync

    print(f"[split, fp32 tiles] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
    A, B = normal((M, K), 33), normal((K, N), 34)
    A[3, 7] = np.inf
    A[130, 9] = np.nan
    A[200, 11] = np.finfo(np.float32).min
    B[11, :64] = 0
    A[257, 11] = 2.0 ** 60
    A[300] *= np.float32(2.0 ** -120)
    A[301] = (A[301] * np.float32(2.0 ** -126)) * np.float32(2.0 ** -10)
    A[400] = 0
    B[20, 5] = np.inf
    dA, dB = Dev.of(A.T if ta else A), Dev.of(B.T if tb else B)
    dc = Dev(M * N)
    hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, dA.ptr, M if ta else K, dB.ptr, K if tb else N, dc.ptr, N, None), "gemm")
    sync()
    got = dc.get((M, N))
    rows = [0, 3, 129, 130, 131, 200, 257, 300, 301, 400, M - 1]
    with np.errstate(all="ignore"):
        want = A[rows].astype(np.float64) @ B.astype(np.float64)
        mag = np.abs(A[rows].astype(np.float64)) @ np.abs(B.astype(np.float64))
        f32 = want.astype(np.float32)
    g = got[rows]
    assert np.array_equal(np.isnan(g), np.isnan(f32)), "NaNs"
    assert np.array_equal(np.isinf(g), np.isinf(f32)), "infinities"
    fine = np.isfinite(f32)
    # one term at a time in fp32; products of subnormals round to the subnormal grid
    tol = K * 2.0 ** -24 * mag + K * 2.0 ** -149
    assert np.all(np.abs(g[fine].astype(np.float64) - want[fine]) <= tol[fine])
    zeros = got[400][np.arange(N) != 5]
    assert not np.any(zeros) and not np.any(np.signbit(zeros))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("scale", [0, 50])
def test_split_nan_operands(ta, tb, scale):
    # NaNs alone stay on the bf16 instructions (scale 0); beside sums past their range (2^100) the tile does not
    from gpu_util import Dev, hip, hip_check, sync

    for M, N, K in TILES:
        print(f"[split, NaN] ta={ta} tb={tb} {M}x{N}x{K} scale={scale}", flush=True)
        s = np.float32(2.0 ** scale)
        A, B = normal((M, K), 51) * s, normal((K, N), 52) * s
        rows, cols = [0, M // 2, M - 1], [5, N - 1]
        for r in rows:
            A[r, (7 * r) % K] = np.nan
        B[K - 1, cols] = np.nan
        a, b = (np.ascontiguousarray(A.T) if ta else A), (np.ascontiguousarray(B.T) if tb else B)
        da, db, dc = Dev.of(a), Dev.of(b), Dev(M * N)
        hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, a.shape[1], db.ptr, b.shape[1], dc.ptr, N, None), "gemm")
        sync()
        got = dc.get((M, N))
        nan = np.zeros((M, N), bool)
        nan[rows], nan[:, cols] = True, True
        assert np.array_equal(np.isnan(got), nan)
        i, j, want, mag = _sample(np.nan_to_num(a), np.nan_to_num(b), ta, tb, np.random.default_rng(1), M, N)
        fine = ~nan[np.ix_(i, j)]
        tol = K * 2.0 ** -24 * mag if scale else _bound(K, mag)
        assert np.all(np.abs(got[np.ix_(i, j)][fine] - want[fine]) <= tol[fine])


@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 0, 4224, 4224, 96), (1, 0, 4100, 4100, 96), (0, 1, 2050, 1410, 642),
                                         (1, 0, 2048, 1408, 640), (1, 0, 769, 769, 16383), (1, 0, 1531, 777, 1999),
                                         (0, 0, 1024, 4096, 2048), (0, 0, 520, 4100, 2050)])  # the last two: fp32
def test_split_entry_points(oracle, ta, tb, M, N, K):
    # the plain, the fused, the allocation-free, the column-sum and the batched call: one product, without a
    # workspace, and the epilogue the separate kernels' bits
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    print(f"[split entries] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
    a, b = normal((K, M) if ta else (M, K), 35), normal((N, K) if tb else (K, N), 36)
    lda, ldb = a.shape[1], b.shape[1]
    da, db, ref, new = Dev.of(a), Dev.of(b), Dev(M * N), Dev(M * N)
    bias, mask = Dev.of(normal(N, 37)), Dev.of(normal((M, N), 38))
    hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, ref.ptr, N, None), "gemm")
    sync()
    want = ref.get()
    assert hip.ts_hip_gemm_workspace_floats(M, N, K) == 0

    def same(what):
        sync()
        assert_bits_equal(new.get(), want, what)
        new.put(np.full(M * N, np.nan, np.float32))

    hip_check(hip.ts_hip_gemm_noalloc(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, new.ptr, N, None), "noalloc")
    same("noalloc")
    hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, None, 0, None, new.ptr, N, None, 0,
                                    None), "fused")
    same("fused")
    dims, zero = (SZ * 1)(1), (SZ * 1)(0)
    for rank in (0, 1):
        hip_check(hip.ts_hip_gemm_batched(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, new.ptr, N, rank, dims, zero,
                                          zero, M * N, None), "batched")
        same(f"a batch of one, rank {rank}")
    if not tb:
        cs = Dev(N)
        cneed = hip.ts_hip_gemm_colsum_workspace_floats(ta, M, N, K)
        cws = Dev(max(cneed, 2))
        hip_check(hip.ts_hip_gemm_colsum(ta, M, N, K, da.ptr, lda, db.ptr, ldb, new.ptr, N, cs.ptr, cws.ptr, cneed,
                                         None), "colsum")
        same("colsum")
        assert_bits_equal(cs.get(), oracle.sum_dim0_chunked(b), "column sums vs the oracle's order")
    hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, bias.ptr, 1, mask.ptr, new.ptr, N,
                                    None, 0, None), "fused epilogue")
    hip_check(hip.ts_hip_bias_add(ref.ptr, bias.ptr, ref.ptr, M, N, 0, None), "bias")
    hip_check(hip.ts_hip_relu(ref.ptr, ref.ptr, M * N, None), "relu")
    hip_check(hip.ts_hip_relu_backward(mask.ptr, ref.ptr, ref.ptr, M * N, None), "mask")
    sync()
    assert_bits_equal(new.get(), ref.get(), "epilogue")


@pytest.mark.parametrize("ta,tb,batches,M,N,K", [(0, 0, 6, 1024, 1000, 300), (0, 1, 64, 256, 256, 512),
                                                 (1, 0, 5, 700, 900, 1001), (0, 0, 64, 512, 128, 512)])
def test_split_batched(ta, tb, batches, M, N, K):
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    print(f"[split batched] ta={ta} tb={tb} {batches} x {M}x{N}x{K}", flush=True)
    a = normal((batches,) + ((K, M) if ta else (M, K)), 39)
    b = normal((N, K) if tb else (K, N), 40)  # shared by the batch
    a[1, 3, 5] = np.inf  # one row of tiles of one batch to the fp32 instructions
    da, db, dc = Dev.of(a), Dev.of(b), Dev(batches * M * N)
    dims, sa, sb = (SZ * 1)(batches), (SZ * 1)(M * K), (SZ * 1)(0)
    hip_check(hip.ts_hip_gemm_batched(ta, tb, M, N, K, da.ptr, a.shape[2], db.ptr, b.shape[1], dc.ptr, N, 1, dims, sa,
                                      sb, M * N, None), "batched")
    sync()
    got = dc.get((batches, M, N))
    for i in (0, 1, batches - 1):
        A = (a[i].T if ta else a[i]).astype(np.float64)
        B = (b.T if tb else b).astype(np.float64)
        with np.errstate(all="ignore"):
            want = A @ B
            mag = np.abs(A) @ np.abs(B)
        fine = np.isfinite(want)
        assert np.array_equal(np.isfinite(got[i]), fine)
        assert np.all(np.abs(got[i][fine] - want[fine]) <= (K * 2.0 ** -24 * mag)[fine])


@pytest.mark.parametrize("ta,tb", [(1, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("left", [1, 2, 3])
def test_split_last_rows_stay_inside(ta, tb, left):
    # a last tile of one to three rows, K in whole stages: what lies behind an operand is not read (an
    # infinity there would send the tile to the fp32 instructions)
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    M = N = 1152 + left
    K = 1024
    print(f"[split, last rows] ta={ta} tb={tb} 2 x {M}x{N}x{K}", flush=True)
    a, b = normal((K, M) if ta else (M, K), 43), normal((N, K) if tb else (K, N), 44)
    dims, shared = (SZ * 1)(2), (SZ * 1)(0)
    out = []
    for behind in (0.0, np.inf):
        tail = np.full(8, behind, np.float32)
        da, db = Dev.of(np.concatenate([a.ravel(), tail])), Dev.of(np.concatenate([b.ravel(), tail]))
        dc = Dev(2 * M * N)
        hip_check(hip.ts_hip_gemm_batched(ta, tb, M, N, K, da.ptr, a.shape[1], db.ptr, b.shape[1], dc.ptr, N, 1, dims,
                                          shared, shared, M * N, None), "batched")
        sync()
        out.append(dc.get((2, M, N)))
    assert_bits_equal(out[1], out[0], "zeros and infinities behind the operands")
    i, j, want, mag = _sample(a, b, ta, tb, np.random.default_rng(1), M, N)
    assert np.all(np.abs(out[0][1][np.ix_(i, j)] - want) <= _bound(K, mag))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("side", ["a", "b"])
def test_split_transformed_operands(ta, tb, side):
    # an elementwise chain applied as the operand is loaded: the bits of a buffer that holds its values, also
    # where a tile is left to the fp32 instructions, and with the column sums
    import ctypes

    from gpu_util import Dev, hip, hip_check, sync
    from test_xf_gpu import OTHER, _apply, _xf

    for M, N, K in TILES:
        print(f"[split, transformed] ta={ta} tb={tb} {side} {M}x{N}x{K}", flush=True)
        assert hip.ts_hip_gemm_takes_xf(ta, tb, M, N, K, 0) == 1
        a, b = normal((K, M) if ta else (M, K), 53), normal((N, K) if tb else (K, N), 54)
        a.flat[7], b.flat[11], b.flat[-1] = np.inf, np.nan, 2.0 ** 100  # the last one squared: an infinity
        ax, bx = (_apply(a, OTHER), b) if side == "a" else (a, _apply(b, OTHER))
        x = ctypes.byref(_xf(OTHER))
        xa, xb = (x, None) if side == "a" else (None, x)
        lda, ldb = a.shape[1], b.shape[1]
        da, db, dax, dbx = Dev.of(a), Dev.of(b), Dev.of(ax), Dev.of(bx)
        got, want = Dev(M * N), Dev(M * N)
        hip_check(hip.ts_hip_gemm_fused_xf(ta, tb, M, N, K, da.ptr, lda, xa, db.ptr, ldb, xb, None, 0, None, got.ptr,
                                           N, None, 0, None), "fused_xf")
        hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, dax.ptr, lda, dbx.ptr, ldb, want.ptr, N, None), "gemm")
        sync()
        assert_bits_equal(got.get(), want.get(), f"{M}x{N}x{K}")
        if ta and not tb:
            cs_got, cs_want = Dev(N), Dev(N)
            hip_check(hip.ts_hip_gemm_colsum_xf(ta, M, N, K, da.ptr, lda, xa, db.ptr, ldb, xb, got.ptr, N, cs_got.ptr,
                                                None, 0, None), "colsum_xf")
            hip_check(hip.ts_hip_gemm_colsum(ta, M, N, K, dax.ptr, lda, dbx.ptr, ldb, want.ptr, N, cs_want.ptr, None,
                                             0, None), "colsum")
            sync()
            assert_bits_equal(got.get(), want.get(), f"{M}x{N}x{K} with column sums")
            assert_bits_equal(cs_got.get(), cs_want.get(), "column sums")
