"""The output head over vocabularies at the edges of its kernels' splits.  The logits (2 rows a wave,
8192 a round of the launch) row by row against the oracle; the top-N picks (128 slices, 2048
keys a round of a block: fewer tokens than slices, a ragged last slice, one token more than a
round a slice) exact against a stable sort of the logits of the same call.  Runs through the C
ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxg
import qxo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [32, 37, 129, 4099, 128 * 2048 + 1])
def test_topn(vocab):
    m = qxg.MemModel(1, vocab, 8, True, True, seed=3)
    c = qxg.Context(0)
    try:
        c.load(m.path, verify=False)
        x = np.random.default_rng(vocab).standard_normal(2048).astype(np.float32)
        for n in (1, 8, 32):
            _, lg, ids, vals = c.final_head(x, n)
            want = np.argsort(-lg, kind="stable")[:n]   # equal logits: the lower token first
            assert np.array_equal(ids, want) and np.array_equal(vals, lg[want].astype(np.float64))
            _, lg, ids, vals = c.final_head(0 * x, n)   # all equal
            assert not lg.any() and np.array_equal(ids, np.arange(n)) and not vals.any()
    finally:
        c.close()
        m.close()


def test_topn_keeps_the_sign_of_zero(tmp_path):
    """Head rows with negative block scales give logits of -0 on a zero residual; the picks carry the
    logits' own bits, in the order of the indexes, -0 and +0 being equal."""
    p, vocab = tmp_path / "m.qxf", 4099
    qxg.generate_model(p, layers=1, vocab=vocab, experts=8, seed=3)
    data = np.memmap(p, np.uint8, "r+")
    count, at = int(data[16:20].view(np.uint32)[0]), int(data[24:32].view(np.uint64)[0])
    for i in range(count):
        e = data[at + 208 * i:at + 208 * (i + 1)]
        if bytes(e[:96]).split(b"\0")[0] == b"output.weight":
            offset, size = (int(v) for v in e[144:160].view(np.uint64))
            blocks = data[offset:offset + size].reshape(vocab, 8, 210)
            blocks[::3, :, 192:208] = 1                                      # positive scales in a block,
            blocks[::3, :, 208:210] = np.array([0x8400], np.uint16).view(np.uint8)   # times -2^-14
    c = qxg.Context(0)
    try:
        c.load(p, verify=False)
        _, lg, ids, vals = c.final_head(np.zeros(2048, np.float32), 32)
        assert not lg.any() and np.signbit(lg).any() and not np.signbit(lg).all()
        assert np.array_equal(ids, np.arange(32)) and np.array_equal(np.signbit(vals), np.signbit(lg[:32]))
    finally:
        c.close()


@pytest.mark.parametrize("vocab", [1, 7, 8191, 8192, 8193, 16385, 3 * 8192 - 1])
def test_logits_of_every_round(vocab):
    m = qxg.MemModel(0, vocab, 8, False, True, seed=3)
    c, om = qxg.Context(0), qxo.Model(m.path)
    try:
        c.load(m.path, verify=False)
        x = np.random.default_rng(vocab).standard_normal(2048).astype(np.float32)
        _, lg, _, _ = c.final_head(x, 1)
        _, want, _, _ = om.final_head(x, vocab, 1)
        # a row's error: 64 f32 sums of exact products and their tree, some 2^-24 each of values no
        # larger than 10 times the rows' root mean square: within 1e-5 of the latter
        assert np.abs(lg - want).max() <= 1e-5 * np.sqrt(np.mean(want.astype(np.float64) ** 2))
    finally:
        om.close()
        c.close()
        m.close()
