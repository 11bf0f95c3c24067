"""Batched prefill where its result could hang on more than the inputs, or lose bits that a norm
over whole rows does not show: calls repeated bit for bit, attention heads whose context comes
from small weights or small V scales alone, scores near and beyond f32's range, SwiGLU far in its tail.
Models are generated files with a few tensors rewritten, so that the part in question stands
alone in the output; the oracle reads the same files.  Runs through the C ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxg
import qxo
from helpers import REL_L2, rel_l2, seeded_kv

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qxg.Context(0)
    yield c
    c.close()


def tensors(path):
    """{name: (dims, writable bytes)} of a QXF1 file."""
    data = np.memmap(path, np.uint8, "r+")
    count, at = int(data[16:20].view(np.uint32)[0]), int(data[24:32].view(np.uint64)[0])
    found = {}
    for i in range(count):
        e = data[at + 208 * i:at + 208 * (i + 1)]
        dims, (offset, size) = e[112:144].view(np.uint64), e[144:160].view(np.uint64)
        found[bytes(e[:96]).split(b"\0")[0].decode()] = ([int(v) for v in dims], data[int(offset):int(offset + size)])
    return found


def one_layer(path, **kw):
    qxg.generate_model(path, layers=1, vocab=256, experts=16, embedding=False, head=False, **kw)
    return tensors(path)


def oracle_q(om, x, pos):
    """The roped q heads [32, 128] of one residual row (in double)."""
    w = lambda name: om.tensor("blk.0." + name)[2].view(np.float32).astype(np.float64)
    xd = x.astype(np.float64)
    xn = (xd / np.sqrt((xd * xd).mean() + 1e-6) * w("attn_norm.weight")).astype(np.float32)
    q = qxo.matvec(23, om.tensor("blk.0.attn_q.weight")[2], 4096, 2048, xn).reshape(32, 128).astype(np.float64)
    q = q / np.sqrt((q * q).mean(1, keepdims=True) + 1e-6) * w("attn_q_norm.weight")
    angle = pos * 1e6 ** (-np.arange(64) / 64)
    c, s = np.cos(angle), np.sin(angle)
    return np.concatenate([q[:, :64] * c - q[:, 64:] * s, q[:, :64] * s + q[:, 64:] * c], 1)


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


def kv_head_model(path, kv):
    """A layer whose attention output is what kv head `kv`'s eight q heads contribute (the O
    matrix's blocks of other heads scaled by 0) and whose own V rows are 0."""
    t = one_layer(path, seed=29)
    o = t["blk.0.attn_output.weight"][1].reshape(2048, 16, 136)
    o[:, np.arange(16) // 4 != kv, :2] = 0
    t["blk.0.attn_v.weight"][1].reshape(-1, 136)[:, :2] = 0


def attention_rows(ctx, path, om, p0, x, rows):
    """Each row's distance from the oracle's over the same cache rows."""
    n = len(x)
    ctx.load(path, verify=False)
    ctx.kv_create(1, p0 + n)
    ctx.kv_write(0, 0, *rows)
    fi, _, _ = ctx.prefill_layer(0, p0, x)
    okv = qxo.KV(1, p0 + n)
    okv.k[0], okv.v[0], okv.ks[0], okv.vs[0] = ctx.kv_read(0, 0, p0 + n)
    return [rel_l2(fi[t], x[t] + qxo.attention_layer_given_row(om, 0, p0 + t, okv, x[t])[0]) for t in range(n)]


@pytest.mark.parametrize("n,lead", [(1, 12), (3, 18), (3, 40)])
def test_attention_behind_a_sink(ctx, tmp_path, n, lead):
    """A first position whose score leads by `lead` holds zeros, so that the context is what a later
    chunk of the same wave adds with weights of e^-lead."""
    p, p0, kv = tmp_path / "m.qxf", 200, 1
    kv_head_model(p, kv)
    om = qxo.Model(p)
    x = np.random.default_rng(7 + n).standard_normal((n, 2048)).astype(np.float32)
    k, v, ks, vs = seeded_kv(41, p0)
    q = np.concatenate([oracle_q(om, x[t], p0 + t)[8 * kv:8 * kv + 8] for t in range(n)])
    row = np.linalg.lstsq(q, np.ones(len(q)), rcond=None)[0]   # the shortest row with the same score for all of them
    codes = np.round(row / np.abs(row).max() * 127)
    k[0, 128 * kv:128 * kv + 128] = codes
    ks[0] = lead * np.sqrt(128) / (q @ codes).mean()
    v[:] = 0   # (other heads too: the context row is packed under one scale)
    v[128:160, 128 * kv:128 * kv + 128] = np.random.default_rng(5).integers(-127, 128, (32, 128))
    vs *= np.float32(np.exp(lead))
    errs = attention_rows(ctx, p, om, p0, x, (k, v, ks, vs))
    om.close()
    assert max(errs) <= REL_L2, errs


@pytest.mark.parametrize("scale", [1e-2, 1e-4, -1e-4])
def test_attention_after_zero_v_scales(ctx, tmp_path, scale):
    """Whole chunks of V scales 0 (as unwritten positions hold), then small ones (or negative ones, which
    a cache may be given)."""
    p, p0, kv = tmp_path / "m.qxf", 250, 2
    kv_head_model(p, kv)
    om = qxo.Model(p)
    x = 1e-3 * np.random.default_rng(9).standard_normal((2, 2048)).astype(np.float32)
    k, v, ks, vs = seeded_kv(43, p0)
    vs[:128] = 0
    vs[128:] *= scale * 127
    errs = attention_rows(ctx, p, om, p0, x, (k, v, ks, vs))
    om.close()
    assert max(errs) <= REL_L2, errs


@pytest.mark.parametrize("scale", [1.0, 0.9 * 2.0 ** 60])
def test_attention_large_scores(ctx, tmp_path, scale):
    """Scores near 2^70, and one of a query and a K scale that are each far inside f32's range while their
    product is not: finite in the oracle's double, it outweighs every other position.  A non-finite K
    scale's score is 0."""
    p, p0, kv = tmp_path / "m.qxf", 70, 0
    kv_head_model(p, kv)
    t = tensors(p)
    t["blk.0.attn_q_norm.weight"][1].view(np.float32)[:] = 2.0 ** 64
    om = qxo.Model(p)
    x = np.random.default_rng(11).standard_normal((1, 2048)).astype(np.float32)
    k, v, ks, vs = seeded_kv(47, p0)
    q = oracle_q(om, x[0], p0)[8 * kv:8 * kv + 8]
    row = np.linalg.lstsq(q, np.ones(8), rcond=None)[0]
    k[40, 128 * kv:128 * kv + 128] = np.round(row / np.abs(row).max() * 127)
    ks[40] = scale
    ks[3] = np.nan
    ks[4] = np.inf
    errs = attention_rows(ctx, p, om, p0, x, (k, v, ks, vs))
    om.close()
    assert max(errs) <= REL_L2, errs


@pytest.mark.parametrize("n", [1, 20])
def test_swiglu_tail(ctx, tmp_path, n):
    """Every gate value about -88, where 1 + e^-gate is beyond the range whose reciprocal is a
    normal f32: silu is near 5e-37 and still counts, the up rows being large."""
    p = tmp_path / "m.qxf"
    t = one_layer(p, seed=31)
    x = np.random.default_rng(13).standard_normal(2048).astype(np.float32)
    t["blk.0.ffn_gate_inp.weight"][1].view(np.float32)[:] *= np.float32(1e-3)   # keep several experts' weights
    gate = t["blk.0.ffn_gate_exps.weight"][1].reshape(-1, 8 * 74)
    gate[:] = gate[0].copy()
    up = t["blk.0.ffn_up_exps.weight"][1].reshape(-1, 74)
    up[:, :2] = np.array([0x7400], np.uint16).view(np.uint8)   # fp16 16384
    norm = t["blk.0.ffn_norm.weight"][1].view(np.float32)
    norm[:] = 1
    om = qxo.Model(p)
    xd = x.astype(np.float64)
    g = qxo.matvec(17, np.array(gate[0]), 1, 2048, (xd / np.sqrt((xd * xd).mean() + 1e-6)).astype(np.float32))[0]
    x = (x * -np.sign(g)).astype(np.float32)
    norm[:] = 88.0 / abs(g)
    y, want, _, _ = om.moe_layer(0, x)
    om.close()
    assert 0 < np.abs(want).max() < 1e-20
    t["blk.0.attn_output.weight"][1].reshape(-1, 136)[:, :2] = 0   # the expert half's input is x itself
    ctx.load(p, verify=False)
    ctx.kv_create(1, 32)
    fi, moe, _ = ctx.prefill_layer(0, 0, np.tile(x, (n, 1)))
    assert np.array_equal(fi, np.tile(x, (n, 1)))
    # e^88 times an error of the gate's f32 sum, 1e-6 of it at most, is 88 times as much of the result
    for r in range(n):
        assert rel_l2(moe[r], want) <= 88e-6, (r, rel_l2(moe[r], want))
