"""A call that fails has waited for the work that it queued: the launches read the context's pinned
input, which the next call overwrites.  The failure is an error left over in the HIP runtime, put
there from the host.  Runs through the C ABI (include/qxg.h)."""
import ctypes
import time

import numpy as np
import pytest

import qxg

pytestmark = pytest.mark.gpu


def test_failed_call_waits():
    with open("/proc/self/maps") as maps:
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64.so" in line))
    m = qxg.MemModel(16, 4096, 128, True, True, seed=5)
    c = qxg.Context(0)
    try:
        c.load(m.path, verify=False)
        c.kv_create(16, 512)
        prompt = np.random.default_rng(3).integers(0, 4096, 512).astype(np.uint32)
        _, want, _, _, ms = c.prefill(prompt, want_logits=True)
        assert ms > 2   # device time of the work below
        hip.hipSetDevice(1 << 20)   # refused; the error stays until it is asked for
        with pytest.raises(qxg.QxgError, match="launch"):
            c.prefill(prompt)
        start = time.perf_counter()
        c.kv_read(0, 0, 1)   # waits for the stream
        assert time.perf_counter() - start < 1e-3
        assert np.array_equal(c.prefill(prompt, want_logits=True)[1], want)
    finally:
        c.close()
        m.close()
