"""The mean loss and the correct count of softmax cross-entropy over many rows: the row terms are
added by 1024 threads, ceil(B / 1024) rows each in order, and a tree over the threads."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from orcaml_amd import _lib

pytestmark = pytest.mark.gpu


def f32_tree(x, B):
    """The kernel's own order in f32."""
    per = -(-B // 1024)
    s = np.zeros(1024, np.float32)
    for k in range(per):
        r = np.arange(1024) * per + k
        s[r < B] = s[r < B] + x[r[r < B]]
    w = 512
    while w:
        s[:w] = s[:w] + s[w:2 * w]
        w //= 2
    return s[0]


@pytest.mark.parametrize("B", [1, 1023, 1024, 1025, 4093, 4096, 4100, 5000, 8192, 8190])
def test_mean_loss_and_count_over_many_rows(ctx, B):
    C = 5
    rng = np.random.default_rng(B)
    logits = rng.standard_normal((B, C)).astype(np.float32) * 2
    labels = rng.integers(0, C, B).astype(np.int32)
    dl, dlab = ctx.upload(logits), ctx.upload(labels)
    loss, correct, preds = ctx.alloc(4), ctx.alloc(8), ctx.alloc(4 * B)
    _lib.call("orca_hip_softmax_ce", ctx.handle, dl.ptr, B, C, None, dlab.ptr, loss.ptr, None, preds.ptr, correct.ptr)
    assert correct.download(np.int64, 1)[0] == int((np.argmax(logits, 1) == labels).sum())
    np.testing.assert_array_equal(preds.download(np.int32, B), np.argmax(logits, 1))
    # each row's own loss, from the same kernel on one row: the mean over B = 1 is the row's term
    rows = np.empty(B, np.float32)
    one, pick = ctx.alloc(4), np.unique(np.linspace(0, B - 1, 64).astype(int))
    x = logits.astype(np.float64)
    term = np.log(np.exp(x - x.max(1, keepdims=True)).sum(1)) + x.max(1) - x[np.arange(B), labels]
    for r in pick:
        _lib.call("orca_hip_softmax_ce", ctx.handle, dl.ptr + 4 * C * int(r), 1, C, None, dlab.ptr + 4 * int(r), one.ptr,
                  None, None, None)
        assert abs(one.download(count=1)[0] - term[r]) <= 1e-6 * max(1.0, abs(term[r]))
    # the mean: rows exact to 1e-6, B f32 additions on top of the kernel's order of the rounded terms
    rows[:] = term
    want = f32_tree(rows, B) * np.float32(1.0 / B)
    assert abs(loss.download(count=1)[0] - want) <= 2e-6 * abs(want) + 1e-7
