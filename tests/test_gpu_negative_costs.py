"""Guided jobs in which more pixels are resolved than there were to resolve:
inpainting a smaller part of an image, or redoing everything after a random
initialisation. The guide's weight (alpha (1 - resolved / to resolve))^3 is
negative there, so costs can be, partial sums do not only grow, and the
reference's rule (a candidate is dropped as soon as a partial sum reaches the
best cost so far) is more than the least cost. Every path against the oracle,
bit for bit."""
import pytest

import tsgpu as ts
from oracle import refcpu as R
from tests.test_gpu_flow import team
from tests.test_gpu_parity import assert_same, run_pair
from tests.test_gpu_serve import same
from tsgpu import synth

pytestmark = pytest.mark.gpu

PATHS = [team(1), team(2), team(4), team(8), dict(flow=0), dict(ahead=0), dict(flow=0, persist=1, defer=1),
         dict(prefetch_max=40, flow_head=16, team_waves=80)]


def inpainting(w, h, n):
    exs = [synth.example(700 + i, w, h) for i in range(n)]
    gds = [synth.blobs(710 + i, w, h) for i in range(n)]
    return exs, gds, synth.blobs(720, w, h), synth.ellipse_mask(721, w, h)


def inpaint_pair(exs, gds, tg, mk, seed, k, m, tune):
    h, w = mk.shape[:2]
    rest = len(exs) - 1
    job = R.Job(R.default_params(seed=seed, nearest_neighbors=k, random_sample_locations=m), exs, w, h, example_guides=gds,
                target_guide=tg, inpaint_mask=mk, inpaint_color=exs[0], inpaint_index=0, sample_kind=[2] + [0] * rest,
                sample_masks=[mk] + [None] * rest)
    job.run(threads=8, **ts.default_schedule())
    b = ts.Session.builder().seed(seed).nearest_neighbors(k).random_sample_locations(m).load_target_guide(tg)
    b.inpaint_example(mk, ts.Example(exs[0]).with_guide(gds[0]).set_sample_method(mk), ts.Dims(w, h))
    for e, g in zip(exs[1:], gds[1:]):
        b.add_example(ts.Example(e).with_guide(g))
    return b.build().set_tuning(**tune).run(), job


@pytest.mark.parametrize("tune", PATHS)
@pytest.mark.parametrize("n,k,m", [(1, 50, 50), (2, 20, 33), (2, 64, 100)])
def test_guided_inpainting(ctx, tune, n, k, m):
    gen, job = inpaint_pair(*inpainting(70, 56, n), seed=n + k, k=k, m=m, tune=tune)
    assert gen.resolved_score.min() < 0.0  # costs below zero did occur
    assert_same(gen, job)


@pytest.mark.parametrize("tune", PATHS)
def test_everything_redone_after_random_init(ctx, tune):
    exs = [synth.example(730 + i, 44 + 5 * i, 40) for i in range(3)]
    gds = [synth.blobs(735 + i, 44 + 5 * i, 40) for i in range(3)]
    gen, job = run_pair(exs, 40, 36, seed=3, example_guides=gds, target_guide=synth.blobs(739, 40, 36), random_init=60,
                        backtrack_percent=1.0, backtrack_stages=3, tuning=tune)
    assert_same(gen, job)


def test_together(ctx):
    def build():
        exs, gds, tg, mk = inpainting(90, 64, 1)
        b = ts.Session.builder().seed(2).load_target_guide(tg)
        b.inpaint_example(mk, ts.Example(exs[0]).with_guide(gds[0]).set_sample_method(mk), ts.Dims(90, 64))
        return b.build()

    alone = build().run()
    for whole in (True, False):
        batch = ts.Batch(ctx)
        tickets = [batch.submit(build()) for _ in range(3)]
        if whole:
            batch.run_all()
        while batch.step(1):
            pass
        for t in tickets:
            assert same(batch.take(t), alone)
        batch.close()
