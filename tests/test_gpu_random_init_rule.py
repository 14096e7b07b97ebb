"""Random initialisation of few points (the moved entries in a map) and of more
than one pixel in 128 (the whole list), on both sides of that line, up to every
pixel, against the oracle; pick orders on the device and on the host. Bit for
bit."""
import pytest

from tests.test_gpu_parity import assert_same, run_pair
from tsgpu import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("n", [16, 17, 18, 2303, 2304])  # 64 x 36 = 2304 = 18 * 128
def test_map_and_list(ctx, n, flow):
    gen, job = run_pair([synth.example(60, 33, 29)], 64, 36, seed=n, random_init=n, backtrack_stages=2,
                        nearest_neighbors=12, random_sample_locations=9, tuning=dict(flow=flow))
    assert_same(gen, job)
