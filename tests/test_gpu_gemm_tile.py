"""The small-tile products (T x T tiles, T = 16, 32, 64) and the pipelined 128-tile product on
operands that are not 16-byte aligned, each tile forced in turn: exact on integers in every
layout, at the edges of tiles and slabs, with and without a K split, through padded leading
dimensions and bases off by one float (NaN in the padding and beyond the operand: nothing read
there may reach C), with the exact column sum and every epilogue."""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from oracle import oracle as O
from orcaml_amd import _lib
from tests.util import int_matrix

pytestmark = pytest.mark.gpu


def context(**switches):
    """A context created under ORCA_HIP_GEMM_<name>=<value>."""
    from orcaml_amd.device import Context

    names = {f"ORCA_HIP_GEMM_{k}": v for k, v in switches.items()}
    old = {k: os.environ.get(k) for k in names}
    os.environ.update(names)
    try:
        return Context(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


@pytest.fixture(scope="module", params=["16/1", "32/1", "64/1", "128/1", "16/2", "32/3", "64/2", "128/3"])
def tctx(request):
    """A context whose products take one tile (and K split)."""
    tile, splits = request.param.split("/")
    c = context(TILE=tile, SPLITS=splits)
    yield c
    c.close()


class Operand:
    """A rows x cols matrix on the device with `pad` extra floats per row and `shift` floats in
    front, NaN wherever it has no value."""

    def __init__(self, ctx, a, pad, shift):
        rows, self.ld = a.shape[0], a.shape[1] + pad
        host = np.full(shift + (rows - 1) * self.ld + a.shape[1] + 64, np.nan, np.float32)
        view = np.lib.stride_tricks.as_strided(host[shift:], a.shape, (4 * self.ld, 4))
        view[:] = a
        self.buf = ctx.upload(host)
        self.ptr = self.buf.ptr + 4 * shift


def product(ctx, ta, tb, A, B, pad=0, shift=0, colsum=False, kind=_lib.EPI_NONE, bias=None, mask=None, pre=False):
    (M, K), N = A.shape, B.shape[1]
    a = Operand(ctx, np.ascontiguousarray(A.T) if ta else A, pad, shift)
    b = Operand(ctx, np.ascontiguousarray(B.T) if tb else B, pad, shift)
    ldc = N + pad
    c = ctx.upload(np.full(M * ldc, 7.0, np.float32))
    keep = [ctx.upload(x) for x in (bias, mask) if x is not None]
    e = _lib.Epilogue(kind)
    if bias is not None:
        e.bias = keep[0].ptr
    if mask is not None:
        e.mask, e.ldmask = keep[-1].ptr, N
    p = ctx.upload(np.full(M * ldc, 7.0, np.float32)) if pre else None
    if pre:
        e.pre = p.ptr
    cs = ctx.alloc(4 * N) if colsum else None
    if colsum:
        e.colsum = cs.ptr
    _lib.call("orca_hip_gemm", ctx.handle, int(ta), int(tb), M, N, K, a.ptr, a.ld, b.ptr, b.ld, c.ptr, ldc,
              ctypes.byref(e))
    out = c.download(count=M * ldc).reshape(M, ldc)
    np.testing.assert_array_equal(out[:, N:], np.full((M, pad), 7.0, np.float32))
    res = [np.ascontiguousarray(out[:, :N])]
    if pre:
        res.append(np.ascontiguousarray(p.download(count=M * ldc).reshape(M, ldc)[:, :N]))
    if colsum:
        res.append(cs.download(count=N))
    return res


# M, N, K: one element past, at and short of each tile; K from less than a slab to several, whole
# and ragged; the fewest floats the kernels take.
SHAPES = [(17, 17, 17), (16, 32, 64), (15, 33, 255), (31, 65, 257), (64, 128, 784), (63, 129, 513), (129, 127, 300),
          (132, 260, 36), (1, 18, 4), (4, 20, 1000), (20, 4, 131), (200, 26, 333), (130, 70, 1030),
          (70, 130, 31), (129, 65, 32), (66, 131, 33)]  # around half of a one-slab 64-tile


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_every_tile_exact_on_integers(tctx, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 13 + K)
    A, B = int_matrix(rng, (M, K)), int_matrix(rng, (K, N))
    want = (A.astype(np.int64) @ B.astype(np.int64)).astype(np.float32)
    sums = O.sum_to_shape(B, (1, N)).reshape(N)
    for pad, shift in ((0, 0), (4, 0), (3, 1), (1, 2)):
        for ta, tb in ((False, False), (False, True), (True, False), (True, True)):
            for colsum in (False, True) if not tb else (False,):
                got = product(tctx, ta, tb, A, B, pad, shift, colsum)
                np.testing.assert_array_equal(got[0], want, err_msg=f"{ta} {tb} {pad} {shift}")
                if colsum:
                    np.testing.assert_array_equal(got[1], sums, err_msg=f"{ta} {tb} {pad} {shift}")


@pytest.mark.parametrize("M,N,K", [(33, 65, 257), (128, 64, 512), (130, 70, 300), (128, 256, 96)])
def test_every_tile_epilogues_and_column_sum_bits(tctx, M, N, K):
    """Real data: each epilogue is the composed ops on the tile's own product, bit for bit, and the
    column sum has the bits of sum_to_shape."""
    rng = np.random.default_rng(M + N + K)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    bias, mask = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    mask[::5, ::3] = 0.0
    prod, cs = product(tctx, False, False, A, B, colsum=True)
    np.testing.assert_array_equal(cs, O.sum_to_shape(B, (1, N)).reshape(N))
    # any order of a K-term f32 sum is within K 2^-24 sum |a b|
    bound = K * 2.0 ** -24 * (np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64)))
    assert (np.abs(prod - A.astype(np.float64) @ B.astype(np.float64)) <= bound).all()
    biased = O.add(prod, O.expand(bias.reshape(1, N), (M, N)))
    masked = O.relu_backward(prod, mask)
    np.testing.assert_array_equal(product(tctx, False, False, A, B, kind=_lib.EPI_BIAS, bias=bias)[0], biased)
    np.testing.assert_array_equal(product(tctx, False, False, A, B, kind=_lib.EPI_BIAS_RELU, bias=bias)[0],
                                  O.relu(biased))
    np.testing.assert_array_equal(product(tctx, False, False, A, B, kind=_lib.EPI_RELU_MASK, mask=mask)[0], masked)
    for kind, kw, got, kept in ((_lib.EPI_BIAS_RELU_PRE, {"bias": bias}, O.relu(biased), biased),
                                (_lib.EPI_RELU_MASK_PRE, {"mask": mask}, masked, prod)):
        c, p = product(tctx, False, False, A, B, kind=kind, pre=True, **kw)
        np.testing.assert_array_equal(c, got)
        np.testing.assert_array_equal(p, kept)


@pytest.mark.parametrize("batch,M,N,K", [(5, 40, 24, 70), (3, 197, 197, 64), (260, 9, 8, 33),
                                           (3, 130, 70, 130),  # 18 64-tiles, six an entry, in three slabs
                                           (3, 70, 66, 32)])  # half of a slab
def test_every_tile_batched(tctx, batch, M, N, K):
    from orcaml_amd.backend import HipBackend

    rng = np.random.default_rng(batch + K)
    A, B = int_matrix(rng, (batch, M, K)), int_matrix(rng, (batch, K, N))
    want = (A.astype(np.int64) @ B.astype(np.int64)).astype(np.float32)
    be = HipBackend(tctx)
    At, Bt = (np.ascontiguousarray(x.transpose(0, 2, 1)) for x in (A, B))
    for x, y in ((A, B), (None, B), (A, None), (None, None)):
        a = be.from_f32_slice((batch, M, K), A) if x is not None else be.transpose(
            be.from_f32_slice((batch, K, M), At), (batch, K, M), 1, 2)
        b = be.from_f32_slice((batch, K, N), B) if y is not None else be.transpose(
            be.from_f32_slice((batch, N, K), Bt), (batch, N, K), 1, 2)
        got = be.to_f32_vec(be.matmul(a, b, (batch, M, K), (batch, K, N))).reshape(batch, M, N)
        np.testing.assert_array_equal(got, want)


def test_forced_split_of_many_entries_stays_within_the_grid():
    """64 chunks of each of 1100 entries would be 70400 layers of the grid."""
    from orcaml_amd.backend import HipBackend

    ctx = context(TILE="64", SPLITS="64")
    be = HipBackend(ctx)
    rng = np.random.default_rng(2)
    A, B = int_matrix(rng, (1100, 4, 4096), -1, 2), int_matrix(rng, (1100, 4096, 4), -1, 2)
    a, b = be.from_f32_slice(A.shape, A), be.from_f32_slice(B.shape, B)
    got = be.to_f32_vec(be.matmul(a, b, A.shape, B.shape)).reshape(1100, 4, 4)
    np.testing.assert_array_equal(got, A @ B)
    del a, b, be
    ctx.close()


@pytest.mark.parametrize("batch,m,k,n", [(3, 33, 20, 65), (5, 197, 64, 197), (7, 70, 300, 40), (2, 16, 5, 18), (9, 130, 70, 31),
                                           (13, 330, 64, 330), (21, 260, 64, 260)])
def test_batched_tiles_in_any_number(ctx, batch, m, k, n):
    """Tile counts that are no multiple of the eight XCDs, each operand transposed in turn; the last two
    on 64-tiles, 468 and 525 of them, whose order follows the XCDs."""
    from orcaml_amd.backend import HipBackend

    ctx.prof_reset()
    ctx.prof_enable(True)
    rng = np.random.default_rng(batch * m + n)
    be = HipBackend(ctx)
    A, B = int_matrix(rng, (batch, m, k), -3, 4), int_matrix(rng, (batch, k, n), -3, 4)
    for ta, tb in ((0, 0), (1, 0), (0, 1)):
        a = be.from_f32_slice((batch, k, m) if ta else (batch, m, k), np.ascontiguousarray(A.swapaxes(1, 2)) if ta else A)
        b = be.from_f32_slice((batch, n, k) if tb else (batch, k, n), np.ascontiguousarray(B.swapaxes(1, 2)) if tb else B)
        a = be.transpose(a, (batch, k, m), 1, 2) if ta else a
        b = be.transpose(b, (batch, n, k), 1, 2) if tb else b
        out = np.asarray(be.to_f32_vec(be.matmul(a, b, (batch, m, k), (batch, k, n)))).reshape(batch, m, n)
        np.testing.assert_array_equal(out, A @ B)
    ctx.prof_enable(False)
    if m > 250 and ctx.prof_report()["num_cus"] == 256:
        assert all("_t64" in name["name"] for name in ctx.prof_report()["kernels"] if name["name"].startswith("gemm_"))


@pytest.mark.parametrize("ta,M,N,K,tiles", [
    # the column sum's chain of adds is longer than any product: the product still takes its own cheapest tile
    (True, 2560, 48, 2942, (32, 64)), (True, 105, 920, 3316, (32, 64)), (True, 96, 1160, 2968, (32, 64)),
    # one round of 128-tiles against four and more one-slab 64-tiles a CU
    (False, 2290, 1128, 10, (64,)), (False, 1064, 1960, 17, (64,)), (False, 3648, 1000, 16, (64,))])
def test_tile_of_lopsided_products(ctx, ta, M, N, K, tiles):
    if ctx.prof_report()["num_cus"] != 256:
        pytest.skip("tile counts chosen for 256 compute units")
    rng = np.random.default_rng(M + N)
    A, B = int_matrix(rng, (M, K), -3, 4), int_matrix(rng, (K, N), -3, 4)
    ctx.prof_reset()
    ctx.prof_enable(True)
    got = product(ctx, ta, False, A, B, kind=_lib.EPI_NONE if ta else _lib.EPI_RELU_MASK,
                  mask=None if ta else np.ones((M, N), np.float32))[0]
    ctx.prof_enable(False)
    want = A.astype(np.float64) @ B.astype(np.float64)
    np.testing.assert_array_equal(got, want.astype(np.float32))
    names = {k["name"].split()[0] for k in ctx.prof_report()["kernels"]}
    kernel = "gemm_tn" if ta else "gemm_nn"
    assert any(n in (f"{kernel}_t{t}", f"{kernel}_t{t}_ua") for n in names for t in tiles), names


def test_more_rows_than_grid_rows_of_small_tiles(ctx):
    """2^21 + 3 rows: 32-row tiles, the cheapest for this width and a K of one of their slabs and two of
    the 64-tiles', would need 65537 grid rows; 100 rows less and they are taken."""
    rng = np.random.default_rng(5)
    A, B = int_matrix(rng, ((1 << 21) + 3, 68), -2, 3), int_matrix(rng, (68, 20), -2, 3)
    a, b, c = ctx.upload(A), ctx.upload(B), ctx.alloc(A.shape[0] * 80)
    for rows, tile in ((A.shape[0] - 100, "_t32"), (A.shape[0], "_t64")):
        ctx.prof_reset()
        ctx.prof_enable(True)
        _lib.call("orca_hip_gemm", ctx.handle, 0, 0, rows, 20, 68, a.ptr, 68, b.ptr, 20, c.ptr, 20, None)
        ctx.prof_enable(False)
        if ctx.prof_report()["num_cus"] == 256:
            assert any(f"gemm_nn{tile}_ua" in k["name"] for k in ctx.prof_report()["kernels"])
    np.testing.assert_array_equal(c.download(count=A.shape[0] * 20).reshape(-1, 20), A @ B)


@pytest.mark.parametrize("switches,kernel", [
    ({"TILE": "16"}, "gemm_nn_t16"), ({"TILE": "128"}, "gemm_nn_pipe"), ({"SMALL_TILES": "0"}, "gemm_nn_pipe"),
    # the generic kernel's tile, and values that name no tile: the cost rule's choice for the others
    ({"TILE": "128x64"}, "gemm_nn_t32"), ({"TILE": "128x128"}, "gemm_nn_t32"), ({"TILE": "64abc"}, "gemm_nn_t32"),
    ({"TILE": "128x64", "FAST": "0"}, "gemm_nn"), ({"TILE": "128x128", "FAST": "0"}, "gemm_nn")])
def test_tile_switches(switches, kernel):
    ctx = context(**switches)
    if ctx.prof_report()["num_cus"] != 256:
        pytest.skip("tile counts chosen for 256 compute units")
    rng = np.random.default_rng(1)
    A, B = int_matrix(rng, (256, 1024)), int_matrix(rng, (1024, 1024))
    ctx.prof_reset()
    ctx.prof_enable(True)
    got = product(ctx, False, False, A, B)[0]
    ctx.prof_enable(False)
    np.testing.assert_array_equal(got, (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32))
    names = {k["name"].split()[0] for k in ctx.prof_report()["kernels"]}
    assert kernel in names, names
    ctx.close()
