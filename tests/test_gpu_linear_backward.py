"""A hidden layer's two backward products from one grid (the trainer's small layers): every
gradient against an fp64 backward pass, at sizes that take each of the tile pairs, aligned and
odd, with the bias gradient from the grid's own blocks and from the head."""
from __future__ import annotations

import numpy as np
import pytest

from orcaml_amd.mlp import MLPTrainer
from tests.util import int_matrix

pytestmark = pytest.mark.gpu


def backward64(dims, params, x, labels):
    hs, h, L = [x.astype(np.float64)], x.astype(np.float64), len(dims) - 1
    for l in range(L):
        h = h @ params[2 * l].astype(np.float64) + params[2 * l + 1]
        if l + 1 < L:
            h = np.maximum(h, 0)
            hs.append(h)
    e = np.exp(h - h.max(1, keepdims=True))
    d = e / e.sum(1, keepdims=True)
    d[np.arange(len(labels)), labels] -= 1
    d /= len(labels)
    grads = [None] * (2 * L)
    for l in range(L - 1, -1, -1):
        grads[2 * l], grads[2 * l + 1] = hs[l].T @ d, d.sum(0, keepdims=True)
        if l:
            d = (d @ params[2 * l].astype(np.float64).T) * (hs[l] > 0)
    return grads


@pytest.mark.parametrize("dims,batch,pairs", [
    ((64, 128, 128, 10), 64, {"t16_t16"}), ((24, 19, 21, 5), 3, {"t16_t16_ua"}),
    ((100, 1024, 1024, 10), 256, {"t32_t64"}), ((50, 1001, 333, 26), 200, {"t32_t32_ua", "t16_t16_ua"}),
    ((20, 257, 129, 33, 20), 65, {"t16_t16_ua"}), ((16, 300, 40, 64, 18), 130, {"t16_t16_ua"}),
    ((32, 900, 1100, 10), 250, {"t32_t64_ua"}), ((8, 36, 2000, 40), 64, {"t16_t16", "t32_t32"}),
    ((20, 1933, 680, 10), 568, {"t64_t64_ua"}), ((24, 1308, 252, 10), 576, {"t64_t64"}),
    ((20, 904, 40, 10), 640, {"t32_t16"}), ((20, 167, 121, 10), 674, {"t32_t16_ua"})])
def test_gradients_of_paired_products(ctx, dims, batch, pairs):
    if ctx.prof_report()["num_cus"] != 256:
        pytest.skip("tile counts chosen for 256 compute units")
    rng = np.random.default_rng(sum(dims) + batch)
    # small integers scaled by powers of two: the forward pass is exact, so the ReLU masks are
    params = []
    for i, o in zip(dims[:-1], dims[1:]):
        params += [int_matrix(rng, (i, o), -1, 2) * np.float32(2.0 ** -4), int_matrix(rng, (1, o), -2, 3) * np.float32(0.25)]
    x = int_matrix(rng, (batch, dims[0]), 0, 3)
    labels = rng.integers(0, dims[-1], batch).astype(np.int32)
    tr = MLPTrainer(ctx, dims, batch, kind="sgd", lr=0.0)
    tr.set_params(params)
    tr.set_batch(x, labels=labels)
    ctx.prof_reset()
    ctx.prof_enable(True)
    tr.step()
    ctx.prof_enable(False)
    names = {k["name"].split()[0] for k in ctx.prof_report()["kernels"]}
    assert {n.replace("gemm_linear_bw_", "") for n in names if n.startswith("gemm_linear_bw_")} == pairs, names
    for i, (got, want) in enumerate(zip(tr.grads(), backward64(dims, params, x, labels))):
        # f32 sums of at most max(batch, width) terms per layer, the logits exact
        err = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
        assert err < 5e-6, (i, err)
    tr.close()
