"""Batched prefill at the edges of its tiles, one layer replayed on the GPU's own inputs
against the oracle (each row on its own at 1e-5).  Runs through the C ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxo
import qxg
from helpers import REL_L2, rel_l2, seeded_kv

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
@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 64, 65, 97, 128, 129, 160])
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
    for t in sorted({0, 14, 15, 16, 30, 31, 32, 33, 63, 64, 95, 96, 127, 128, n - 2, n - 1} & set(range(n))):
        y, m, _, _ = om.moe_layer(layer, fi[t])
        assert rel_l2(moe[t], m) <= REL_L2, (t, rel_l2(moe[t], m))
        assert rel_l2(out[t], y) <= REL_L2, (t, rel_l2(out[t], y))
    om.close()


@pytest.mark.parametrize("mix,layer", [(0, 0), (1, 1)])
@pytest.mark.parametrize("n", [1, 8, 32, 33, 64, 65, 128, 129, 257])
def test_dense_row_tiles_and_parts(ctx, models, mix, layer, n):
    """Q/K/V and O at the edges of their row tiles, which are also where the number of parts of K
    changes (8 and 16 parts up to 64 rows, 4 and 8 up to 128, ...): the attention half of the
    edge rows against the oracle over the GPU's own cache rows, IQ4_XS and Q5_K V and O."""
    p = models / f"m{mix}.qxf"
    ctx.load(p)
    layers = 4 if mix else 1
    ctx.kv_create(layers, 300)
    x = np.random.default_rng(70 + n).standard_normal((n, 2048)).astype(np.float32)
    x[n // 2] *= 1e3
    fi, _, _ = ctx.prefill_layer(layer, 0, x)
    okv = qxo.KV(layers, 300)
    okv.k[layer, :n], okv.v[layer, :n], okv.ks[layer, :n], okv.vs[layer, :n] = ctx.kv_read(layer, 0, n)
    om = qxo.Model(p)
    for t in sorted({0, 31, 32, 63, 64, 127, 128, 255, 256, n // 2, n - 1} & set(range(n))):
        a, _, _, rk, rv, (sk, sv) = qxo.attention_layer_given_row(om, layer, t, okv, x[t])
        assert rel_l2(fi[t], x[t] + a) <= REL_L2, (t, rel_l2(fi[t], x[t] + a))
        assert np.abs(okv.k[layer, t].astype(int) - rk.astype(int)).max() <= 1, t
        assert np.abs(okv.v[layer, t].astype(int) - rv.astype(int)).max() <= 1, t
    om.close()


@pytest.mark.parametrize("n,p0,odd", [(1, 0, 0), (1, 31, 0), (3, 127, 0), (5, 128, 0), (4, 290, 0), (13, 260, 1), (66, 70, 1)])
def test_attention_runs_and_scales(ctx, models, n, p0, odd):
    """Attention over one and several runs of positions (several from 256 positions on while the
    tokens are few), chunks that hold only masked positions for some token, and, with odd, V
    scales 1e6 apart inside a chunk and between chunks and a NaN K scale (the reference's scores
    of that position are 0): every row against the oracle over the same cache rows."""
    p = models / "m0.qxf"
    ctx.load(p)
    ctx.kv_create(1, 400)
    okv = qxo.KV(1, 400)
    if p0:
        k, v, ks, vs = seeded_kv(300 + p0, p0)
        if odd:
            vs[::7] *= 1e-6
            vs[40:44] *= 1e3
            ks[11] = np.nan
        ctx.kv_write(0, 0, k, v, ks, vs)
        okv.k[0, :p0], okv.v[0, :p0], okv.ks[0, :p0], okv.vs[0, :p0] = k, v, ks, vs
    x = np.random.default_rng(31 + n).standard_normal((n, 2048)).astype(np.float32)
    fi, _, _ = ctx.prefill_layer(0, p0, x)
    okv.k[0, p0:p0 + n], okv.v[0, p0:p0 + n], okv.ks[0, p0:p0 + n], okv.vs[0, p0:p0 + n] = ctx.kv_read(0, p0, n)
    om = qxo.Model(p)
    for t in range(n):
        a = qxo.attention_layer_given_row(om, 0, p0 + t, okv, x[t])[0]
        assert rel_l2(fi[t], x[t] + a) <= REL_L2, (t, rel_l2(fi[t], x[t] + a))
    om.close()
