"""Device-to-host reads on both sides of the staged path's threshold, into fresh, reused and
odd-addressed memory, after work still queued on the stream, and from two contexts in two threads."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from orcaml_amd import _lib
from orcaml_amd.device import Context

pytestmark = pytest.mark.gpu

M = 1 << 20


@pytest.mark.parametrize("n", [1, 8 * M - 4, 8 * M, 8 * M + 4, 16 * M + 4, 32 * M - 4, 32 * M, 37 * M + 12])
def test_read_back_exact(ctx, n):
    rng = np.random.default_rng(n)
    x = rng.integers(0, 255, n, dtype=np.uint8)
    buf = ctx.upload(x)
    for shift in (0, 1, 4):
        host = np.full(n + shift + 8, 0xAB, np.uint8)
        _lib.call("orca_hip_d2h", ctx.handle, host.ctypes.data + shift, buf.ptr, n)
        np.testing.assert_array_equal(host[shift:shift + n], x)
        assert (host[:shift] == 0xAB).all() and (host[shift + n:] == 0xAB).all()


def test_read_follows_queued_work_and_two_threads(ctx):
    def work(c, value, out):
        n = 5 * M  # floats
        buf = c.alloc(4 * n)
        for k in range(20):
            c.fill(buf, value + k, n)  # the read below must wait for the last of these
        out.append(buf.download(count=n))

    other, got = Context(0), ([], [])
    threads = [threading.Thread(target=work, args=(c, v, g)) for c, v, g in ((ctx, 1.0, got[0]), (other, 100.0, got[1]))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, v in zip(got, (20.0, 119.0)):
        np.testing.assert_array_equal(g[0], np.float32(v))
    other.close()
