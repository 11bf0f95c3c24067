"""The output head's top-N picks over vocabularies at the edges of their split (128 slices, 2048
keys a round of a block): fewer tokens than slices, a ragged last slice, one token more than a
round a slice.  Exact against a stable sort of the logits of the same call.  Runs through the C
ABI (include/qxg.h)."""
import numpy as np
import pytest

import qxg

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
