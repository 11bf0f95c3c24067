"""The prefill's own layout of the attention matrices: made by the first batched prefill after a
bind and by nothing else, made anew for another model, and not needed where it does not fit.
Runs through the C ABI (include/qxg.h)."""
import ctypes

import numpy as np
import pytest

import qxg
from helpers import rel_l2

pytestmark = pytest.mark.gpu

PLANES = 16 * (5120 * 2048 + 2048 * 4096) * 9 // 8   # of 16 layers of the benchmark formats


class Hip:
    def __init__(self):
        with open("/proc/self/maps") as maps:
            self.lib = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64.so" in line))

    def free(self):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def take(self, size):
        p = ctypes.c_void_p()
        status = self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size))
        self.lib.hipGetLastError()
        return p if status == 0 else None

    def give(self, p):
        assert self.lib.hipFree(p) == 0


@pytest.fixture(scope="module")
def models():
    ms = [qxg.MemModel(16, 4096, 16, True, True, seed=s) for s in (3, 4)]
    yield ms
    for m in ms:
        m.close()


def test_only_batched_prefill_makes_the_planes(models):
    c, hip = qxg.Context(0), Hip()
    try:
        c.load(models[0].path, verify=False)
        c.kv_create(16, 64)
        bound = hip.free()
        c.generate([1, 2, 3], 4)
        c.set_activation("q8_k_compat")
        c.prefill(np.arange(20, dtype=np.uint32))
        c.set_activation("f32")
        assert bound - hip.free() < PLANES // 4
        c.prefill(np.arange(20, dtype=np.uint32))
        used = hip.free()
        assert bound - used >= PLANES
        c.prefill(np.arange(20, dtype=np.uint32))
        assert hip.free() == used
        c.load(models[1].path, verify=False)   # given back with the model they were made from
        assert hip.free() - used >= PLANES * 3 // 4
    finally:
        c.close()


def test_planes_follow_the_model(models):
    prompt = np.random.default_rng(2).integers(0, 4096, 40).astype(np.uint32)

    def logits(*paths):
        c = qxg.Context(0)
        try:
            for path in paths:
                c.load(path, verify=False)
                c.kv_create(16, 64)
                lg = c.prefill(prompt, want_logits=True)[1]
            return lg
        finally:
            c.close()

    assert np.array_equal(logits(models[0].path, models[1].path), logits(models[1].path))


def test_prefill_without_room_for_the_planes(models):
    """With less free memory than the planes take, the prompt goes by token steps, and as
    before once there is room again."""
    prompt = np.random.default_rng(6).integers(0, 4096, 40).astype(np.uint32)
    c, hip = qxg.Context(0), Hip()
    taken = []
    try:
        c.load(models[0].path, verify=False)
        c.kv_create(16, 64)
        c.generate([1, 2, 3], 4)
        c.set_layer_path(0)
        c.generate([1, 2, 3], 4)
        c.set_layer_path(1)
        taken.append(hip.take(hip.free() - PLANES))
        for _ in range(64):   # until the planes do not fit (there is more than the free memory reported)
            p = hip.take(PLANES)
            if not p:
                break
            hip.give(p)
            taken.append(hip.take(PLANES // 8))
        assert not p and all(taken)
        _, steps, _, _, _ = c.prefill(prompt, want_logits=True)
        while taken:
            hip.give(taken.pop())
        free = hip.free()
        _, batched, _, _, _ = c.prefill(prompt, want_logits=True)
        assert free - hip.free() >= PLANES
        assert rel_l2(steps, batched) <= 1e-3
        assert not np.array_equal(steps, batched)   # (two ways of summing)
    finally:
        for p in taken:
            hip.give(p)
        c.close()
