"""softmax and its backward along the last axis (the row kernels) at the edges
of their column ranges, bit for bit against the oracle's loops."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from conftest import assert_bits_equal, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [
    (130, 9), (70, 10), (9, 33), (9, 64), (8, 65), (17, 128), (7, 129), (8, 256), (3, 257), (5, 512), (4, 513), (6, 1000),
    (1, 1024), (5, 1025), (3, 2048), (5, 2049), (5, 4097), (3, 8192), (3, 8193), (2, 16385), (1, 32768), (2, 32769),
    (2050, 2049), (2049, 3001), (3601, 4097), (1801, 8200), (901, 16385), (9, 40000)])
def test_softmax_rows(rows, cols):
    from gpu_util import Dev, hip, hip_check, sync

    print(f"[softmax rows] {rows}x{cols}", flush=True)
    x = normal((rows, cols), cols, 4.0)
    x[0, cols // 2] = -np.inf  # masked out
    x[-1, -1] = np.finfo(np.float32).min
    dx, dy = Dev.of(x), Dev(x.size)
    hip_check(hip.ts_hip_softmax(dx.ptr, dy.ptr, rows, cols, 1, None), "softmax")
    sync()
    y = dy.get(x.shape)
    assert_bits_equal(y, O.softmax(x, 1), "softmax")
    go = normal((rows, cols), cols + 1)
    dgo, dgi = Dev.of(go), Dev(x.size)
    hip_check(hip.ts_hip_softmax_backward(dy.ptr, dgo.ptr, dgi.ptr, rows, cols, 1, None), "softmax_backward")
    sync()
    assert_bits_equal(dgi.get(x.shape), O.softmax_bwd(y, go, 1), "softmax_backward")


def test_softmax_rows_without_a_value():
    # rows of NaN, of -inf alone and with +inf: the loops' NaNs where they give them
    from gpu_util import Dev, hip, hip_check, sync

    x = normal((5, 100), 3)
    x[0, :] = -np.inf
    x[1, 7] = np.nan
    x[2, 50] = np.inf
    x[3, :] = np.nan
    dx, dy = Dev.of(x), Dev(x.size)
    hip_check(hip.ts_hip_softmax(dx.ptr, dy.ptr, 5, 100, 1, None), "softmax")
    sync()
    assert_bits_equal(dy.get(x.shape), O.softmax(x, 1), "softmax")


def test_softmax_more_rows_than_a_grid_holds():
    # 2^29 rows of 10 columns and some take 2^32 threads, more than a launch: the rows at both ends and
    # where the launches meet, forward and backward
    from gpu_util import Dev, hip, hip_check, sync

    rows, cols = (1 << 29) + 100, 10
    print(f"[softmax rows] {rows}x{cols}", flush=True)
    n = rows * cols
    dx, dy, dgi = Dev(n), Dev(n), Dev(n)  # 21.5 GB each
    hip_check(hip.ts_hip_fill(dx.ptr, 0.0, n, None), "fill")
    hip_check(hip.ts_hip_fill(dgi.ptr, 7.0, n, None), "fill")
    sync()
    first = ((1 << 32) - 1) // 64 * 8  # rows of the first launch
    windows = [(0, 20), (first - 20, 40), (rows - 20, 20)]
    values = [normal((k, cols), 60 + i, 3.0) for i, (_, k) in enumerate(windows)]

    def put(d, r, v):
        hip_check(hip.ts_hip_memcpy(d.ptr + 4 * r * cols, v.ctypes.data, v.size, 0), "H2D")

    def get(d, r, k):
        out = np.empty((k, cols), np.float32)
        hip_check(hip.ts_hip_memcpy(out.ctypes.data, d.ptr + 4 * r * cols, out.size, 1), "D2H")
        return out

    for (r, _), v in zip(windows, values):
        put(dx, r, v)
    hip_check(hip.ts_hip_softmax(dx.ptr, dy.ptr, rows, cols, 1, None), "softmax")
    hip_check(hip.ts_hip_softmax_backward(dy.ptr, dx.ptr, dgi.ptr, rows, cols, 1, None), "softmax_backward")
    sync()
    for (r, k), v in zip(windows, values):
        y = O.softmax(v, 1)
        assert_bits_equal(get(dy, r, k), y, f"softmax, rows from {r}")
        assert_bits_equal(get(dgi, r, k), O.softmax_bwd(y, v, 1), f"softmax_backward, rows from {r}")
