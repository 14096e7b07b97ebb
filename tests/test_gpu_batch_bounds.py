"""Schedules whose largest batch is not the one of the redo and new-pixel shifts
(a first stage with larger batches, a fixed size above the cap): every buffer
that holds a batch is sized for it, on the paths that keep one (a launch per
batch, the work-queue engine), and the results are the oracle's. Bit for bit."""
import pytest

import tsgpu as ts
from tests.test_gpu_parity import assert_same, run_pair
from tests.test_gpu_serve import same
from tsgpu import synth

pytestmark = pytest.mark.gpu

SCHEDULES = [
    dict(px_per_batch=0, redo_shift=6, new_shift=3, max_batch=0, first_new_shift=1),
    dict(px_per_batch=0, redo_shift=9, new_shift=9, max_batch=700, first_new_shift=1),
    dict(px_per_batch=300, redo_shift=5, new_shift=6, max_batch=5, first_new_shift=7),
]


@pytest.mark.parametrize("sched", SCHEDULES)
@pytest.mark.parametrize("tune", [dict(flow=0, ahead=0), dict(flow=0), dict(flow=1)])
def test_single_job(ctx, sched, tune):
    gen, job = run_pair([synth.example(740, 40, 37)], 92, 64, sched=sched, seed=1, nearest_neighbors=12,
                        random_sample_locations=9, backtrack_stages=2, tuning=tune)
    assert_same(gen, job)


@pytest.mark.parametrize("sched", SCHEDULES)
def test_engine(ctx, sched):
    def build():
        b = ts.Session.builder().seed(1).add_example(synth.example(740, 40, 37)).output_size(ts.Dims(92, 64))
        return b.nearest_neighbors(12).backtrack_stages(2).build().set_schedule(**sched)

    alone = build().run()
    batch = ts.Batch(ctx)
    tickets = [batch.submit(build()) for _ in range(2)]
    while batch.step(1):
        pass
    for t in tickets:
        assert same(batch.take(t), alone)
    batch.close()
