"""Batched prefill at the edges of its tiles, one layer replayed on the GPU's own inputs
against the oracle (each row on its own at 1e-5).  Runs through the C ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxo
import qxg
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qxg.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    for mix in (0, 1):
        qxg.generate_model(d / f"m{mix}.qxf", layers=4 if mix else 1, vocab=256, experts=16, embedding=False, head=False,
                           seed=17, mix=mix)
    return d


@pytest.mark.parametrize("mix,layer", [(0, 0), (1, 1), (1, 2), (1, 3)])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65, 97, 160])
def test_expert_row_tiles(ctx, models, mix, layer, n):
    """n nearly equal rows, so the same eight experts hold about n pairs each: one ragged
    row tile, full tiles, two tiles a pass and several passes of one expert.  The rows at
    the tiles' edges are checked."""
    p = models / f"m{mix}.qxf"
    ctx.load(p)
    ctx.kv_create(4 if mix else 1, 256)
    rng = np.random.default_rng(5 + n)
    x = (rng.standard_normal(2048) + 0.02 * rng.standard_normal((n, 2048))).astype(np.float32)
    fi, moe, out = ctx.prefill_layer(layer, 0, x)
    om = qxo.Model(p)
    for t in sorted({0, 15, 16, 30, 31, 32, 33, 63, 64, 95, 96, 127, 128, n - 2, n - 1} & set(range(n))):
        y, m, _, _ = om.moe_layer(layer, fi[t])
        assert rel_l2(moe[t], m) <= REL_L2, (t, rel_l2(moe[t], m))
        assert rel_l2(out[t], y) <= REL_L2, (t, rel_l2(out[t], y))
    om.close()
