"""Team runs with more than 64 random candidates (k_flow_slice) against the
oracle: slices that leave members a part of a group or more than one, few
neighbours, masks, guides, costs that no candidate beats, the unpruned rule.
Bit for bit."""
import numpy as np
import pytest

import tsgpu as ts
from tests.test_gpu_flow import team
from tests.test_gpu_parity import assert_same, run_pair
from tsgpu import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [2, 4, 8])
@pytest.mark.parametrize("k,m", [(50, 65), (1, 66), (64, 513), (20, 4096)])
def test_slices(ctx, t, k, m):
    n = 24 if m > 1000 else 45
    gen, job = run_pair([synth.example(890 + k, 33, 28)], n, n - 7, seed=m, nearest_neighbors=k, random_sample_locations=m,
                        backtrack_stages=3, tuning=team(t))
    assert_same(gen, job)


@pytest.mark.parametrize("t", [2, 8])
def test_guided_masked_examples(ctx, t):
    exs = [synth.example(880 + i, 40 + 7 * i, 44) for i in range(3)]
    gds = [synth.blobs(883 + i, 40 + 7 * i, 44) for i in range(3)]
    mk = np.full((44, 47, 4), 255, np.uint8)
    mk[:, ::3, 0] = 0
    gen, job = run_pair(exs, 50, 43, seed=8, example_guides=gds, target_guide=synth.blobs(886, 50, 43), random_init=7,
                        sample_kind=[0, 2, 0], sample_masks=[None, mk, None], random_sample_locations=150, tuning=team(t))
    assert_same(gen, job)


@pytest.mark.parametrize("t", [2, 8])
@pytest.mark.parametrize("prm", [
    dict(cauchy_dispersion=0.0),    # NaN cost tables: the unpruned rule
    dict(cauchy_dispersion=1e-30),  # infinite costs
    dict(tiling_mode=True),
])
def test_cost_extremes_and_tiling(ctx, t, prm):
    gen, job = run_pair([synth.example(870, 33, 41)], 42, 40, seed=4, random_sample_locations=90, tuning=team(t), **prm)
    if prm.get("cauchy_dispersion", 1.0) == 0.0:
        assert np.array_equal(gen.coord, job.state()[1])  # NaN scores compare unequal
    else:
        assert_same(gen, job)


def test_single_items_on_two_workgroups(ctx):
    sched = dict(px_per_batch=1, redo_shift=0, new_shift=0, max_batch=0, first_new_shift=0)
    gen, job = run_pair([synth.example(871, 30, 30)], 24, 21, sched=sched, seed=2, random_sample_locations=80,
                        tuning=team(8, flow_wgs=2))
    assert_same(gen, job)


def test_teams_of_several_sizes(ctx):
    m = synth.ellipse_mask(872, 90, 70)
    gen, job = run_pair([synth.example(873, 90, 70)], 90, 70, seed=6, inpaint_mask=m, inpaint_index=0, sample_kind=[2],
                        sample_masks=[m], random_sample_locations=100, backtrack_stages=3,
                        tuning=dict(flow=1, ahead=1, prefetch_max=40, flow_head=16, team_waves=80))
    assert_same(gen, job)
