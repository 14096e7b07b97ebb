"""exp_f32 (texture-synthesis_amd/csrc/exp_dd.h), the unguided wave runs' form of
the neighbour weights' (float)exp(-x): against the host C library on the sweep
arguments of test_exp_sweep.py, on the host (2^24 of them, and the one that the
device's own exp got wrong) and on the device (2^30); the mismatch counts are
zero. test_exp_sweep.py does the same for exp_dd, which every other run uses."""
import numpy as np
import pytest

import tsgpu as ts
from oracle import refcpu as R
from tests.test_exp_sweep import CHUNK, SWEEP


def test_host_matches_the_c_library():
    for i0, n in [(0, 1 << 24), (50710905, 1)]:
        assert R.exp_compare(i0, ts.debug_exp_f32_sweep_host(i0, n)) == (0, (1 << 64) - 1), i0


@pytest.mark.gpu
def test_device_matches_host_over_2e30_arguments(ctx):
    bad = 0
    first = None
    for i0 in range(0, SWEEP, CHUNK):
        n, f = R.exp_compare(i0, ts.debug_exp_f32_sweep(i0, CHUNK, ctx), threads=16)
        if n and first is None:
            first = f
        bad += n
    print(f"device/host exp_f32: {bad} of {SWEEP} differ (first {first})")
    assert bad == 0, (bad, first)


@pytest.mark.gpu
def test_device_and_host_forms_agree(ctx):
    for dev, host in [(ts.debug_exp_sweep, ts.debug_exp_sweep_host), (ts.debug_exp_f32_sweep, ts.debug_exp_f32_sweep_host)]:
        assert np.array_equal(dev(7, 1 << 20, ctx).view(np.uint32), host(7, 1 << 20).view(np.uint32))
