"""On a device with little memory left, jobs run without their stage-ahead sets
instead of failing, alone and in a batch, with the same results. The device is
filled by one allocation of the test's own, which leaves enough for everything
else."""
import ctypes

import numpy as np
import pytest

import tsgpu as ts
from tsgpu import synth

pytestmark = pytest.mark.gpu


class Filled:
    """All but `left` bytes of the device's memory taken, beside what the library holds."""

    def __init__(self, ctx, left):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.p = ctypes.c_void_p()
        ctx.trim()
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        self.n = max(0, free.value - left)

    def __enter__(self):
        if self.n:
            assert self.hip.hipMalloc(ctypes.byref(self.p), ctypes.c_size_t(self.n)) == 0
        return self

    def __exit__(self, *_):
        if self.n:
            assert self.hip.hipFree(self.p) == 0


def build(tiling):
    b = ts.Session.builder().seed(5).add_example(synth.example(750, 64, 64)).tiling_mode(tiling).backtrack_stages(1)
    return b.output_size(ts.Dims(2048, 1800)).build()


def same(a, b):
    return (np.array_equal(a._state, b._state) and np.array_equal(a.resolved_flat, b.resolved_flat)
            and np.array_equal(a.resolved_score.view(np.uint32), b.resolved_score.view(np.uint32)))


def test_jobs_run_without_their_sets(ctx):
    # the sets of such a job take 3.2 GB, everything else 0.3
    want = [build(t).run() for t in (False, True)]
    batch = ts.Batch(ctx)
    batch.set_alone(0, 16 << 30)
    with Filled(ctx, 1 << 30):
        for t, w in zip((False, True), want):
            assert same(build(t).run(), w)
        ticket = batch.submit(build(False))
        batch.run_all()
        assert same(batch.take(ticket), want[0])
    batch.close()
    ctx.trim()
