"""ReLU backward + column sum and the many-parameter optimizer passes at column counts, lengths
and base addresses that are not multiples of 16 bytes: bit for bit the oracle's element-wise results
and the column sums in the kernels' own order, nothing written outside the outputs."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from orcaml_amd import _lib

pytestmark = pytest.mark.gpu


def column_sums(d):
    """64-row chunks in row order, a quarter of the chunks at a time, the quarters in order."""
    chunks = [np.zeros(d.shape[1], np.float32) for _ in range(-(-d.shape[0] // 64))]
    for r in range(d.shape[0]):
        chunks[r // 64] = chunks[r // 64] + d[r]
    per = -(-len(chunks) // 4)
    quarters = []
    for q in range(4):
        s = np.zeros(d.shape[1], np.float32)
        for c in chunks[q * per:(q + 1) * per]:
            s = s + c
        quarters.append(s)
    return ((quarters[0] + quarters[1]) + quarters[2]) + quarters[3]


@pytest.mark.parametrize("rows", [1, 7, 64, 65, 300])
@pytest.mark.parametrize("cols", [1, 3, 4, 5, 6, 7, 8, 333, 1003, 1030])
def test_relu_bw_colsum_any_columns(ctx, rows, cols):
    rng = np.random.default_rng(rows * 31 + cols)
    g, pre = (rng.standard_normal((rows, cols)).astype(np.float32) for _ in range(2))
    pre[rng.random(pre.shape) < 0.1] = 0.0
    want = O.relu_backward(g, pre)
    for shift in (0, 1):
        def put(a):
            return ctx.upload(np.concatenate([np.full(shift, np.nan, np.float32), a.reshape(-1)]))
        dg, dp = put(g), put(pre)
        out = ctx.upload(np.full(shift + rows * cols + 8, 7.0, np.float32))
        cs = ctx.upload(np.full(cols + 4, 7.0, np.float32))
        _lib.call("orca_hip_relu_bw_colsum", ctx.handle, dg.ptr + 4 * shift, dp.ptr + 4 * shift, rows, cols,
                  out.ptr + 4 * shift, cs.ptr)
        got = out.download()[:shift + rows * cols + 8]
        np.testing.assert_array_equal(got[shift:shift + rows * cols].reshape(rows, cols), want)
        assert (got[:shift] == 7.0).all() and (got[shift + rows * cols:] == 7.0).all()
        sums = cs.download()[:cols + 4]
        np.testing.assert_array_equal(sums[:cols], column_sums(want))
        assert (sums[cols:] == 7.0).all()


@pytest.mark.parametrize("kind", ["adamw", "sgd"])
@pytest.mark.parametrize("lens", [(5, 1, 3, 1024, 7, 4), (1030, 2, 4099), (4, 4, 4), (8, 16, 1)])
def test_packed_segments_bit_exact(ctx, kind, lens):
    """Parameters packed without padding, each array at its own odd offset."""
    rng = np.random.default_rng(sum(lens))
    n = sum(lens)
    arrays = [rng.standard_normal(n).astype(np.float32) for _ in range(4)]
    arrays[3] = np.abs(arrays[3])
    shifts = (1, 2, 3, 1)
    bufs = [ctx.upload(np.concatenate([np.full(s, 7.0, np.float32), a, np.full(4, 7.0, np.float32)]))
            for a, s in zip(arrays, shifts)]
    table, off = (_lib.OptSegment * len(lens))(), 0
    for i, length in enumerate(lens):
        p, g, m, v = (b.ptr + 4 * (s + off) for b, s in zip(bufs, shifts))
        table[i] = _lib.OptSegment(p, p, g, m, v, length)
        off += length
    p, g, m, v = (a.copy() for a in arrays)
    if kind == "adamw":
        _lib.call("orca_hip_adamw_multi", ctx.handle, table, len(lens), 1e-3, 0.9, 0.999, 1e-8, 0.01, 3)
        ref = [ctx.upload(a) for a in (p, g, m, v)]  # the flat pass, itself bit-identical to the oracle
        _lib.call("orca_hip_adamw_step", ctx.handle, *(b.ptr for b in ref), n, 1e-3, 0.9, 0.999, 1e-8, 0.01, 3)
        want = [b.download(count=n) for b in ref]
    else:
        _lib.call("orca_hip_sgd_multi", ctx.handle, table, len(lens), 0.1)
        want = [p - g * np.float32(0.1), g, m, v]
    for b, s, w in zip(bufs, shifts, want):
        got = b.download()[:s + n + 4]
        np.testing.assert_array_equal(got[s:s + n], w)
        assert (got[:s] == 7.0).all() and (got[s + n:] == 7.0).all()
