"""The optimizer step in the launch of the first layer's weight gradient (the trainer's small
models): parameters and moments bit for bit from the gradients that the step left behind, by the
same f32 operations in numpy, at sizes that take the different tiles, aligned and odd, with the
first layer's bias gradient from the launch's own blocks and from the head."""
from __future__ import annotations

import math

import numpy as np
import pytest

from orcaml_amd.mlp import MLPTrainer

pytestmark = pytest.mark.gpu
f32 = np.float32


def adamw(p, g, m, v, lr, b1, b2, eps, wd, t):
    m = m * f32(b1) + g * f32(1 - b1)
    v = v * f32(b2) + (g * g) * f32(1 - b2)
    den = np.sqrt(v * f32(1 / (1 - math.pow(b2, t)))) + f32(eps)
    return p * f32(1 - lr * wd) - (m * f32(1 / (1 - math.pow(b1, t)))) / den * f32(lr), m, v


@pytest.mark.parametrize("kind", ["sgd", "adamw"])
@pytest.mark.parametrize("dims,batch", [
    ((784, 128, 128, 10), 64), ((784, 1024, 1024, 10), 256), ((500, 1001, 333, 26), 200), ((1000, 33, 10), 7),
    ((31, 18), 300), ((130, 2050, 70, 20), 40), ((516, 1500, 10), 64), ((5, 19, 3), 1030), ((1021, 1500, 40), 130)])
def test_update_beside_the_first_weight_gradient(ctx, kind, dims, batch):
    rng = np.random.default_rng(sum(dims) + batch)
    lr, b1, b2, eps, wd = 1e-3, 0.9, 0.999, 1e-8, 0.01
    want = []
    for i, o in zip(dims[:-1], dims[1:]):
        want += [(rng.standard_normal((i, o)) / math.sqrt(i)).astype(f32), rng.standard_normal((1, o)).astype(f32) * f32(0.1)]
    tr = MLPTrainer(ctx, dims, batch, kind=kind, lr=lr, weight_decay=wd if kind == "adamw" else 0.0)
    tr.set_params(want)
    m, v = ([np.zeros_like(p) for p in want] for _ in range(2))
    tr.set_batch(rng.random((batch, dims[0]), dtype=f32), labels=rng.integers(0, dims[-1], batch).astype(np.int32))
    for t in range(1, 4):
        ctx.prof_reset()
        ctx.prof_enable(t == 2)
        tr.step()
        ctx.prof_enable(False)
        if t == 2:
            names = [k["name"].split()[0] for k in ctx.prof_report()["kernels"]]
            assert any(n.endswith("_update") for n in names) and kind not in names, names
        for i, g in enumerate(tr.grads()):
            if kind == "adamw":
                want[i], m[i], v[i] = adamw(want[i], g, m[i], v[i], lr, b1, b2, eps, wd, t)
            else:
                want[i] = want[i] - g * f32(lr)
        for got, w in zip(tr.params(), want):
            np.testing.assert_array_equal(got, w)
        if kind == "adamw":
            for which, state in ((0, m), (1, v)):
                for got, w in zip(tr.moments(which), state):
                    np.testing.assert_array_equal(got, w)
    tr.close()


@pytest.mark.parametrize("kind", ["sgd", "adamw"])
def test_update_as_a_pass_of_its_own(ctx, kind, monkeypatch):
    """ORCA_HIP_OVERLAP_UPDATE=0: no update in the weight gradient's launch, the same bits."""
    dims, batch, got = (100, 130, 64, 10), 48, []
    rng = np.random.default_rng(9)
    params = []
    for i, o in zip(dims[:-1], dims[1:]):
        params += [(rng.standard_normal((i, o)) / math.sqrt(i)).astype(f32), rng.standard_normal((1, o)).astype(f32)]
    x, labels = rng.random((batch, dims[0]), dtype=f32), rng.integers(0, 10, batch).astype(np.int32)
    for own in (False, True):
        if own:
            monkeypatch.setenv("ORCA_HIP_OVERLAP_UPDATE", "0")
        tr = MLPTrainer(ctx, dims, batch, kind=kind, lr=1e-2)
        tr.set_params(params)
        tr.set_batch(x, labels=labels)
        ctx.prof_reset()
        ctx.prof_enable(True)
        for _ in range(3):
            tr.step()
        ctx.prof_enable(False)
        names = {k["name"].split()[0] for k in ctx.prof_report()["kernels"]}
        assert any(n.endswith("_update") for n in names) != own and (kind in names) == own, names
        got.append(tr.params())
        tr.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
