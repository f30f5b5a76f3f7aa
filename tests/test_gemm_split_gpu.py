"""Products on the f16 matrix cores (2.2e9 operations and more, 1.5e9 of ragged sizes): every layout at
the edges of the tiles, of the k stages and of the split K, odd leading
dimensions and addresses, the rows that are left to the fp32 instructions, and
one result from every entry point.

Bound, per element: the two factors of a term are each within 2^-24 of
themselves (or 2^-40 of their row's largest, at most 2^-25 of a row that is
split), the smallest partial product left out is below 2^-24 of it, and three
sums of 32 terms are added to a running sum per 32 k, each within two roundings
of 2^-24: 4 + 2 * 3 * K / 32 units of 2^-24 of sum |a| |b|; the fp32 tiles add
one term at a time, K units."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_bits_equal, normal

pytestmark = pytest.mark.gpu

# (trans_a, trans_b, M, N, K, operand pitch pad, operand offset in floats)
CASES = [
    (0, 0, 4224, 4224, 256, 0, 0),      # 256x256 tiles
    (0, 1, 4096, 4096, 256, 0, 0),
    (1, 0, 4096, 4096, 256, 0, 0),
    (1, 1, 4096, 4096, 256, 0, 0),
    (0, 0, 4090, 4093, 225, 0, 1),      # ragged, a partial stage of one k, no aligned address
    (0, 1, 4095, 4091, 255, 3, 1),
    (1, 0, 4093, 4094, 224, 0, 1),
    (1, 1, 4089, 4090, 193, 1, 3),
    (0, 0, 2048, 1408, 640, 0, 0),      # 128x128 tiles, K in two
    (0, 1, 2049, 1409, 641, 0, 0),
    (1, 0, 2051, 1411, 643, 1, 0),
    (1, 1, 2050, 1410, 642, 0, 1),
    (0, 0, 2049, 4097, 200, 0, 0),      # K whole
    (0, 1, 2050, 4099, 191, 1, 1),
    (1, 0, 2051, 4098, 224, 0, 3),
    (1, 1, 2047, 4095, 231, 0, 0),
    (0, 0, 769, 641, 16001, 0, 0),      # few tiles: K split, its last slice short
    (0, 1, 771, 643, 16383, 0, 1),
    (1, 0, 897, 513, 16000, 3, 0),
    (1, 1, 641, 770, 20011, 0, 0),
    (0, 0, 100, 16384, 1024, 0, 0),     # one row of tiles, most of it used
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
    assert np.all(err <= (4 + 6 * (K + 31) // 32) * 2.0 ** -24 * mag)
    # and closer than one rounding a term would leave it, over all
    assert np.sqrt(np.mean(err ** 2)) <= 0.5 * np.sqrt(K) * 2.0 ** -24 * np.sqrt(np.mean(want ** 2))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(4224, 4224, 128), (2048, 1409, 640), (769, 769, 16001)])
def test_split_rows_left_to_fp32(ta, tb, M, N, K):
    # op(A)'s rows: 3 an infinity, 130 a NaN, 200 the type's lowest value beside ordinary ones that meet
    # zeros, 257 one outlier of 2^60, 300 tiny values, 301 subnormals, 400 zeros; op(B)'s column 5 an infinity
    from gpu_util import Dev, hip, hip_check, sync

    print(f"[split, fp32 rows] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
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
    assert np.all(np.abs(g.astype(np.float64) - want)[fine] <= tol[fine])
    assert not np.any(got[400][np.arange(N) != 5])


@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 0, 4224, 4224, 96), (1, 0, 4100, 4100, 96), (0, 1, 2050, 1410, 642),
                                         (1, 0, 2048, 1408, 640), (1, 0, 769, 769, 16383)])
def test_split_entry_points(oracle, ta, tb, M, N, K):
    # the plain, the workspace, the allocation-free and the column-sum call: one product, and the
    # epilogue the separate kernels' bits
    from gpu_util import Dev, hip, hip_check, sync

    print(f"[split entries] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
    a, b = normal((K, M) if ta else (M, K), 35), normal((N, K) if tb else (K, N), 36)
    lda, ldb = a.shape[1], b.shape[1]
    da, db, ref, new = Dev.of(a), Dev.of(b), Dev(M * N), Dev(M * N)
    bias, mask = Dev.of(normal(N, 37)), Dev.of(normal((M, N), 38))
    hip_check(hip.ts_hip_gemm(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, ref.ptr, N, None), "gemm")
    sync()
    want = ref.get()
    need = hip.ts_hip_gemm_workspace_floats(M, N, K)
    assert 0 < need <= 9 << 20
    ws = Dev(need)

    def same(what):
        sync()
        assert_bits_equal(new.get(), want, what)
        new.put(np.full(M * N, np.nan, np.float32))

    hip_check(hip.ts_hip_gemm_noalloc(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, new.ptr, N, None), "noalloc")
    same("noalloc")
    hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, None, 0, None, new.ptr, N, ws.ptr, need,
                                    None), "fused")
    same("workspace")
    if not tb:
        cs = Dev(N)
        cneed = hip.ts_hip_gemm_colsum_workspace_floats(ta, M, N, K)
        cws = Dev(max(cneed, 2))
        hip_check(hip.ts_hip_gemm_colsum(ta, M, N, K, da.ptr, lda, db.ptr, ldb, new.ptr, N, cs.ptr, cws.ptr, cneed,
                                         None), "colsum")
        same("colsum")
        assert_bits_equal(cs.get(), oracle.sum_dim0_chunked(b), "column sums vs the oracle's order")
    hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, bias.ptr, 1, mask.ptr, new.ptr, N,
                                    ws.ptr, need, None), "fused epilogue")
    hip_check(hip.ts_hip_bias_add(ref.ptr, bias.ptr, ref.ptr, M, N, 0, None), "bias")
    hip_check(hip.ts_hip_relu(ref.ptr, ref.ptr, M * N, None), "relu")
    hip_check(hip.ts_hip_relu_backward(mask.ptr, ref.ptr, ref.ptr, M * N, None), "mask")
    sync()
    assert_bits_equal(new.get(), ref.get(), "epilogue")
    new.put(np.full(M * N, np.nan, np.float32))
    hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, None, 0, None, new.ptr, N, None, 0,
                                    None), "no workspace")
    same("the stream-ordered allocator's workspace")
    # one float fewer: the operands scanned by the workgroups, the same scales; one float in all: a K that was split
    # (fewer tiles than CUs) whole, not an error
    new.put(np.full(M * N, np.nan, np.float32))
    args = (ta, tb, M, N, K, da.ptr, lda, db.ptr, ldb, None, 0, None, new.ptr, N, ws.ptr)
    hip_check(hip.ts_hip_gemm_fused(*args, need - 1, None), "a smaller workspace")
    same("a smaller workspace")
    hip_check(hip.ts_hip_gemm_fused(*args, 1, None), "a small workspace")
    if M >= 4096:
        same("a small workspace")
    else:
        sync()
        _, _, _, mag = _sample(a, b, ta, tb, np.random.default_rng(1), M, N)
        assert np.max(np.abs(new.get().astype(np.float64) - want)) <= (8 + 12 * K / 32) * 2.0 ** -24 * np.max(mag)


def test_split_scans_agree():
    # rows and columns of every kind (wide ranges, zeros, infinities, subnormals): the scan's own launch and the
    # workgroups' scan leave the same tiles to the fp32 instructions
    from gpu_util import Dev, hip, hip_check, sync

    rng = np.random.default_rng(7)
    for ta, tb, M, N, K in [(0, 1, 2049, 1025, 1003), (1, 0, 1025, 2051, 1001), (0, 0, 4100, 4100, 131),
                            (1, 1, 1100, 1300, 1999)]:
        print(f"[split scans] ta={ta} tb={tb} {M}x{N}x{K}", flush=True)
        A, B = normal((M, K), 41), normal((K, N), 42)
        A[rng.integers(0, M, 3)] *= np.float32(2.0) ** rng.integers(-60, 60, K).astype(np.float32)
        B[:, rng.integers(0, N, 3)] *= np.float32(2.0) ** rng.integers(-13, 13, (K, 1)).astype(np.float32)
        A[M - 1, K - 1] = np.inf
        A[5] = 0
        A[6] = 1e-42
        B[0, N - 1] = 3e38
        a, b = (np.ascontiguousarray(A.T) if ta else A), (np.ascontiguousarray(B.T) if tb else B)
        da, db, c1, c2 = Dev.of(a), Dev.of(b), Dev(M * N), Dev(M * N)
        need = hip.ts_hip_gemm_workspace_floats(M, N, K)
        ws = Dev(need)
        for c, n in ((c1, need), (c2, need - 1)):
            hip_check(hip.ts_hip_gemm_fused(ta, tb, M, N, K, da.ptr, a.shape[1], db.ptr, b.shape[1], None, 0, None,
                                            c.ptr, N, ws.ptr, n, None), "fused")
        sync()
        assert_bits_equal(c1.get(), c2.get(), f"{M}x{N}x{K}")


@pytest.mark.parametrize("ta,tb,batches,M,N,K", [(0, 0, 6, 1024, 1000, 300), (0, 1, 64, 256, 256, 512),
                                                 (1, 0, 5, 700, 900, 1001), (0, 0, 64, 512, 128, 512)])
def test_split_batched(ta, tb, batches, M, N, K):
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    print(f"[split batched] ta={ta} tb={tb} {batches} x {M}x{N}x{K}", flush=True)
    a = normal((batches,) + ((K, M) if ta else (M, K)), 39)
    b = normal((N, K) if tb else (K, N), 40)  # shared by the batch
    a[1, 3, 5] = np.inf  # one tile of one batch to the fp32 instructions
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
        assert np.all(np.abs(got[i] - want)[fine] <= (K * 2.0 ** -24 * mag)[fine])


@pytest.mark.parametrize("rank", [0, 1])
@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 0, 2048, 1408, 640), (0, 1, 769, 641, 16001), (1, 0, 999, 777, 1001)])
def test_split_batch_of_one(rank, ta, tb, M, N, K):
    # sizes whose 2-D product splits K: the batched call has no room for the partial products
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    print(f"[split, batch of one] ta={ta} tb={tb} {M}x{N}x{K} rank={rank}", flush=True)
    a, b = normal((K, M) if ta else (M, K), 45), normal((N, K) if tb else (K, N), 46)
    da, db, dc = Dev.of(a), Dev.of(b), Dev.of(np.full(M * N, np.nan, np.float32))
    dims, zero = (SZ * 1)(1), (SZ * 1)(0)
    hip_check(hip.ts_hip_gemm_batched(ta, tb, M, N, K, da.ptr, a.shape[1], db.ptr, b.shape[1], dc.ptr, N, rank, dims,
                                      zero, zero, M * N, None), "batched")
    sync()
    got = dc.get((M, N))
    assert np.all(np.isfinite(got))
    i, j, want, mag = _sample(a, b, ta, tb, np.random.default_rng(1), M, N)
    # one fp32 addition per term at most
    assert np.all(np.abs(got[np.ix_(i, j)] - want) <= K * 2.0 ** -24 * mag)


@pytest.mark.parametrize("ta,tb", [(1, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("left", [1, 2, 3])
def test_split_last_rows_stay_inside(ta, tb, left):
    # a last tile of one to three rows, K in whole stages, scanned by the workgroups: what lies behind a
    # row-contiguous operand is not read (an infinity there would send the tile to the fp32 instructions)
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
    assert np.all(np.abs(out[0][1][np.ix_(i, j)] - want) <= (4 + 6 * (K + 31) // 32) * 2.0 ** -24 * mag)
