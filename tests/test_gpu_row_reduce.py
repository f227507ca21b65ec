"""Row reductions ([R, C] -> [R, 1] and whole buffers) on the staged kernel against the oracle's
loops, bit for bit: rows on both sides of a block's 16, columns around slabs of 256 and groups of
four, a base off by one float, special values, and the NaN beyond the buffer that must not be read in."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from orcaml_amd import _lib

pytestmark = pytest.mark.gpu


def reduce(ctx, op, x, out_shape, shift):
    host = np.full(shift + x.size + 64, np.nan, np.float32)
    host[shift:shift + x.size] = x.reshape(-1)
    buf = ctx.upload(host)
    di, ri = _lib.dims(x.shape)
    do, ro = _lib.dims(out_shape)
    out = ctypes.c_void_p()
    _lib.call(f"orca_hip_{op}", ctx.handle, buf.ptr + 4 * shift, di, ri, do, ro, _lib.F32, ctypes.byref(out))
    n = int(np.prod(out_shape))
    got = np.empty(n, np.float32)
    _lib.call("orca_hip_to_f32_vec", ctx.handle, out, n, got.ctypes.data_as(ctypes.c_void_p))
    _lib.call("orca_hip_free", ctx.handle, out)
    return got


def bits(a):
    """The bits of a result, every NaN alike (its payload is the hardware's)."""
    a = np.asarray(a, np.float32).reshape(-1)
    return np.where(np.isnan(a), np.uint32(0x7FC00000), a.view(np.uint32))


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 200])
@pytest.mark.parametrize("cols", [15, 16, 17, 23, 24, 29, 30, 63, 64, 130, 255, 256, 257, 513, 1000, 1030, 1281])
def test_row_reductions_bit_exact(ctx, rows, cols):
    rng = np.random.default_rng(rows * 7 + cols)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x[rng.random(x.shape) < 0.02] = -0.0
    special = x.copy()
    special[rng.random(x.shape) < 0.003] = np.inf
    special[rng.random(x.shape) < 0.003] = -np.inf
    special[rng.random(x.shape) < 0.003] = np.nan
    special[rng.random(x.shape) < 0.01] = np.float32(1e-42)
    special[rows // 2] = -np.inf  # a row whose maximum stays the lowest value
    for a in (x, special):
        for shift in (0, 1):
            np.testing.assert_array_equal(bits(reduce(ctx, "sum_to_shape", a, (rows, 1), shift)),
                                          bits(O.sum_to_shape(a, (rows, 1))))
            np.testing.assert_array_equal(bits(reduce(ctx, "max_to_shape", a, (rows, 1), shift)),
                                          bits(O.max_to_shape(a, (rows, 1))))
            np.testing.assert_array_equal(bits(reduce(ctx, "sum_to_shape", a, (1,), shift)),
                                          bits(O.sum_to_shape(a, (1,))))
    y = x.reshape(rows, 1, cols)
    np.testing.assert_array_equal(bits(reduce(ctx, "sum_to_shape", y, (rows, 1, 1), 0)),
                                  bits(O.sum_to_shape(y, (rows, 1, 1))))


@pytest.mark.parametrize("op", ["sum_to_shape", "max_to_shape"])
def test_many_short_rows_are_not_slower_than_shorter_ones(ctx, op):
    """A thread per row takes about as long for 16 columns as for 15; a staged block per 16 rows took
    1.8 times that (2.2 for a maximum)."""
    rows, best = 1 << 20, {}
    for cols in (15, 16):
        buf = ctx.upload(np.ones(rows * cols, np.float32))
        di, ri = _lib.dims((rows, cols))
        do, ro = _lib.dims((rows, 1))
        times = []
        for _ in range(8):
            out = ctypes.c_void_p()
            ctx.timer_start()
            _lib.call(f"orca_hip_{op}", ctx.handle, buf.ptr, di, ri, do, ro, _lib.F32, ctypes.byref(out))
            times.append(ctx.timer_stop())
            _lib.call("orca_hip_free", ctx.handle, out)
        best[cols] = min(times)
    assert best[16] < 1.45 * best[15], best
