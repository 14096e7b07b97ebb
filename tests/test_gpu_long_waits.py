"""Dependency-ordered runs whose items take long: a wait ends the run only when
nothing of the run moves any more, never for its length."""
import numpy as np
import pytest

import tsgpu as ts
from tsgpu import synth

pytestmark = pytest.mark.gpu


def test_waits_outlast_slow_chains(ctx):
    # a wave per item and 4096 candidates each: the waves furthest ahead wait
    # for thousands of items before theirs
    def run(**tune):
        b = ts.Session.builder().seed(3).random_sample_locations(4096).add_example(synth.example(990, 128, 128))
        return b.output_size(ts.Dims.square(256)).build().set_tuning(**tune).run()

    a, b = run(flow=1, prefetch_max=0), run(flow=0)
    assert np.array_equal(a.image, b.image) and np.array_equal(a.coord, b.coord) and np.array_equal(a.ids, b.ids)
    assert np.array_equal(a.resolved_score.view(np.uint32), b.resolved_score.view(np.uint32))
