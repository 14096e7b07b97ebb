"""The cache of device blocks: cut down on demand, and not a way past a batch's
budget of stage-ahead bytes."""
import numpy as np
import pytest

import tsgpu as ts
from tsgpu import synth

pytestmark = pytest.mark.gpu


def build(side, seed=1):
    b = ts.Session.builder().seed(seed).add_example(synth.example(760, 64, 64)).output_size(ts.Dims.square(side))
    return b.build()


def test_trim(ctx):
    a = build(96).run()
    held = ctx.trim(1 << 62)
    assert held > 96 * 96 * 28  # the job's blocks at least
    assert 0 <= ctx.trim(held // 2) <= held // 2
    assert ctx.trim() == 0
    assert np.array_equal(build(96).run().image, a.image)
    assert ctx.trim(1 << 62) > 0


@pytest.mark.parametrize("tight", [False, True])
def test_larger_blocks_count_whole(ctx, tight):
    # a job's blocks serve requests of half their size and more: a run that
    # would hold more than its budget in them takes blocks of its own sizes
    ctx.trim()

    def run(side, budget):
        batch = ts.Batch(ctx)
        batch.set_alone(0, budget)
        t = batch.submit(build(side))
        batch.run_all()
        g = batch.take(t)
        batch.close()
        return g

    run(256, 1 << 30)
    held = ctx.trim(1 << 62)
    n = 200 * 200
    need = n * 884  # two sets of m = k = 50, their records and pick lists
    got = run(200, int(need * 1.2) if tight else 1 << 30)
    more = ctx.trim(1 << 62) - held
    assert (more > 0.7 * need) if tight else (more < 0.3 * need), (more, need)
    assert np.array_equal(got.image, build(200).run().image)
