"""Broadcast copies and operations by groups of four and reductions over merged axes, at the
shapes where groups, merges and strides end: against numpy."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from conftest import assert_bits_equal, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,out,off", [
    ((8, 1), (8, 1024), 0), ((7, 1), (7, 1023), 0), ((5, 1), (5, 3), 1), ((1,), (1,), 0), ((1, 1, 1), (1, 1, 5), 0),
    ((1, 6, 1, 8), (3, 6, 5, 8), 0), ((3, 1, 5, 1), (3, 7, 5, 9), 2), ((4, 1, 1, 4), (4, 3, 2, 4), 0),
    ((2, 1, 3, 1, 2, 1, 3, 1), (2, 3, 3, 2, 2, 3, 3, 2), 0), ((1, 1, 12), (9, 2, 12), 3), ((1025,), (33, 1025), 0),
    ((2, 3, 4), (2, 3, 4), 0), ((64, 1, 1), (64, 33, 31), 0)])
@pytest.mark.parametrize("scaled", [0, 1])
def test_broadcast_groups(src, out, off, scaled):
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    x = normal(src, 50)
    n = int(np.prod(out))
    dx, dy = Dev.of(x), Dev.of(np.full(n, np.nan, np.float32), offset=off)
    hip_check(hip.ts_hip_broadcast_copy(dx.ptr, (SZ * len(src))(*src), len(src), dy.ptr, (SZ * len(out))(*out), len(out),
                                        ctypes.c_float(0.3), scaled, None), "broadcast_copy")
    sync()
    want = np.ascontiguousarray(np.broadcast_to(x.reshape(src), out))
    assert_bits_equal(dy.get(out), want * np.float32(0.3) if scaled else want)


@pytest.mark.parametrize("shape,mask", [
    ((1, 1, 1), 0b111), ((1, 7, 1), 0b101), ((7, 1, 65), 0b110), ((3, 4, 5, 6), 0b1100), ((3, 4, 5, 6), 0b0110),
    ((3, 4, 5, 6), 0b1010), ((2000, 513), 0b10), ((300, 1, 4097), 0b100), ((70000, 5), 0b10), ((2, 70000, 3), 0b010),
    ((5, 2, 1, 449), 0b1101)])
def test_reduce_merged_axes(shape, mask):
    from gpu_util import Dev, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    x = normal(shape, 51)
    axes = tuple(k for k in range(len(shape)) if (mask >> k) & 1)
    want = x.astype(np.float64).sum(axis=axes)
    mag = np.abs(x.astype(np.float64)).sum(axis=axes)
    dx, dy = Dev.of(x), Dev(max(want.size, 1))
    hip_check(hip.ts_hip_reduce_sum(dx.ptr, (SZ * len(shape))(*shape), len(shape), mask, dy.ptr, ctypes.c_float(0.5), 1,
                                    None), "reduce_sum")
    sync()
    # f64 sums rounded once, then one exact scaling
    err = np.abs(dy.get(want.shape).astype(np.float64) - 0.5 * want)
    assert np.all(err <= 2.0 ** -25 * np.abs(want) * 1.0001 + x.size * 2.0 ** -53 * mag)


@pytest.mark.parametrize("sa,sb,out,off", [
    ((64, 1024), (64, 1), (64, 1024), 0), ((64, 1), (64, 1023), (64, 1023), 0), ((7, 3), (3,), (7, 3), 1),
    ((5, 1), (1, 7), (5, 7), 0), ((1,), (1,), (1, 1), 0), ((4, 1, 6, 1), (3, 1, 8), (4, 3, 6, 8), 0),
    ((2, 3, 4, 5), (3, 1, 5), (2, 3, 4, 5), 2), ((1, 12), (9, 1), (9, 12), 0), ((2, 3, 8), (2, 3, 8), (2, 3, 8), 0),
    ((2, 1, 3, 1, 2, 1, 3, 1), (3, 1, 2, 1, 2, 1, 2), (2, 3, 3, 2, 2, 2, 3, 2), 0), ((1025,), (33, 1), (33, 1025), 0)])
def test_broadcast_binary(sa, sb, out, off):
    from gpu_util import Dev, ZeroIndex, hip, hip_check, sync
    from train_station_amd._ffi import SZ

    a, b = normal(sa, 52), normal(sb, 53)
    b.reshape(-1)[-1] = 0.0  # a zero divisor
    n = int(np.prod(out))
    da, db = Dev.of(a, offset=off), Dev.of(b)
    dims = [(SZ * len(s))(*s) for s in (sa, sb, out)]
    A, B = np.broadcast_to(a, out), np.broadcast_to(b, out)
    with np.errstate(all="ignore"):
        want = [A + B, A - B, A * B, A / B]
    first = int(np.flatnonzero(B.reshape(-1) == 0)[0])
    for op in range(4):
        z = ZeroIndex()
        dy = Dev.of(np.full(n, np.nan, np.float32), offset=off)
        hip_check(hip.ts_hip_broadcast_binary(op, da.ptr, dims[0], len(sa), db.ptr, dims[1], len(sb), dy.ptr, dims[2],
                                              len(out), 0, z.ptr, None), "broadcast_binary")
        sync()
        assert_bits_equal(dy.get(out), np.ascontiguousarray(want[op]), f"op {op}")
        assert z.value() == (first if op == 3 else None)
    z = ZeroIndex()
    hip_check(hip.ts_hip_broadcast_binary(3, da.ptr, dims[0], len(sa), db.ptr, dims[1], len(sb), dy.ptr, dims[2], len(out),
                                          n, z.ptr, None), "unchecked tail")
    sync()
    assert z.value() is None
    bad = (SZ * len(sb))(*[d + 1 for d in sb])
    assert hip.ts_hip_broadcast_binary(0, da.ptr, dims[0], len(sa), db.ptr, bad, len(sb), dy.ptr, dims[2], len(out), 0,
                                       None, None) != 0
