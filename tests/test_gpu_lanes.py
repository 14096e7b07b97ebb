"""Jobs of a batch run whole, several at a time (Batch.run_all, and sessions
that start alone together), against each run by itself. Bit for bit."""
import pytest

import tsgpu as ts
from test_gpu_batch import assert_same_result, build, spec_list
from tsgpu import synth

pytestmark = pytest.mark.gpu


def more_specs():
    d = ts.default_schedule()
    out = spec_list()
    # larger than a lane's team batches, and smaller than one workgroup
    out += [(dict(kind="plain", ex=64, out=o, seed=4600 + o, k=k), d) for o, k in [(9, 5), (200, 50), (251, 20), (300, 50)]]
    return out


# fewer jobs than lanes, as many, more; a budget that holds every buffer, one
# job's at a time, the small jobs' alone, none
@pytest.mark.parametrize("n", [1, 2, 5, 14])
@pytest.mark.parametrize("budget", [None, 1 << 27, 1 << 22, 0])
def test_run_all_equals_each_alone(ctx, n, budget):
    specs = more_specs()[-n:]
    alone = [build(s).run() for s in specs]
    batch = ts.Batch(ctx)
    if budget is not None:
        batch.set_alone(0, budget)
    for _ in range(2):  # the second time on buffers that the first gave back
        tickets = [batch.submit(build(s)) for s in specs]
        batch.run_all()
        assert not any(st for _, st in batch.poll())
        for t, s, a in zip(tickets, specs, alone):
            assert_same_result(batch.take(t), a, f"{s[0]}")
    batch.close()


def test_tuned_jobs_beside_default_ones(ctx):
    # jobs that do not run in dependency order, or keep a set per stage
    tunes = [dict(), dict(flow=0), dict(ahead=0), dict(ahead=2), dict(flow=0, ahead=2), dict(flow_wgs=1)]

    def job(i, **tune):
        s = ts.Session.builder().seed(i).add_example(synth.example(80 + i, 40, 33)).output_size(ts.Dims(70, 61)).build()
        return s.set_tuning(**tune) if tune else s

    alone = [job(i).run() for i in range(len(tunes))]
    batch = ts.Batch(ctx)
    for below in (0, 100):
        batch.set_alone(below, 1 << 30)
        tickets = [batch.submit(job(i, **t)) for i, t in enumerate(tunes)]
        batch.run_all()
        assert not any(st for _, st in batch.poll())
        for i, t in enumerate(tickets):
            assert_same_result(batch.take(t), alone[i], f"{tunes[i]}")
    batch.close()
