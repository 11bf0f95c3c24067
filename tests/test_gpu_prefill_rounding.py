"""Batched prefill where its result could hang on more than the inputs: calls repeated bit for
bit.  Runs through the C ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qxg.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("mix,layer", [(0, 0), (1, 1), (1, 2), (1, 3)])
@pytest.mark.parametrize("n", [80, 300])
def test_calls_repeat(ctx, tmp_path, mix, layer, n):
    """The same call gives the same bits: with 16 experts, 80 tokens are about 40 pairs an expert (a
    full pass and a short one of gate/up and down) and 300 about 150."""
    p = tmp_path / "m.qxf"
    layers = 4 if mix else 1
    qxg.generate_model(p, layers=layers, vocab=256, experts=16, embedding=False, head=False, seed=23, mix=mix)
    ctx.load(p)
    x = np.random.default_rng(n).standard_normal((n, 2048)).astype(np.float32)
    ctx.kv_create(layers, 320)
    first = ctx.prefill_layer(layer, 0, x)
    for _ in range(8):
        again = ctx.prefill_layer(layer, 0, x)
        for name, a, b in zip(("ffn_inp", "moe", "out"), first, again):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (name, np.flatnonzero((a != b).any(1)))
