"""Stages run in dependency order (k_flow_team, k_flow_wave, k_stage_end)
against the oracle, at the sizes where their slices, rounds and rows end:
neighbour counts of a partial row, candidate lists that leave team members
idle or need more rounds than one, batches of one item, every team size, and
stages that redo less, more or all of what is resolved. Bit for bit."""
import numpy as np
import pytest

import tsgpu as ts
from oracle import refcpu as R
from tests.test_gpu_parity import assert_same, run_pair
from tsgpu import synth

pytestmark = pytest.mark.gpu


def team(t, **kw):
    """Every item with a team of t waves (t = 1: a wave per item)."""
    return dict(flow=1, ahead=1, flow_team=t, flow_head_team=t, team_max=t, prefetch_max=1 << 20, **kw)


@pytest.mark.parametrize("t", [1, 2, 4, 8])
@pytest.mark.parametrize("k,m", [(1, 1), (3, 5), (17, 9), (50, 50), (64, 64), (64, 130)])
def test_team_sizes_and_candidate_counts(ctx, t, k, m):
    ex = synth.example(900 + k, 45, 38)
    gen, job = run_pair([ex], 61, 47, seed=k + m, nearest_neighbors=k, random_sample_locations=m, tuning=team(t))
    assert_same(gen, job)


@pytest.mark.parametrize("t", [1, 2, 4, 8])
def test_guided_masked_examples(ctx, t):
    exs = [synth.example(910 + i, 40 + 7 * i, 44) for i in range(3)]
    gds = [synth.blobs(920 + i, 40 + 7 * i, 44) for i in range(3)]
    mk = np.full((44, 47, 4), 255, np.uint8)
    mk[:, ::3, 0] = 0
    gen, job = run_pair(exs, 70, 53, seed=8, example_guides=gds, target_guide=synth.blobs(930, 70, 53), random_init=7,
                        sample_kind=[0, 2, 0], sample_masks=[None, mk, None], tuning=team(t))
    assert_same(gen, job)


@pytest.mark.parametrize("t", [1, 8])
@pytest.mark.parametrize("prm", [
    dict(backtrack_stages=0),
    dict(backtrack_stages=1),
    dict(backtrack_stages=3, backtrack_percent=1.0),   # every stage redoes everything
    dict(backtrack_stages=3, backtrack_percent=0.0),   # empty stages, then all at once
    dict(backtrack_stages=2, backtrack_percent=0.9),
    dict(cauchy_dispersion=0.0),                       # NaN cost tables: the unpruned rule
    dict(cauchy_dispersion=1e-30),                     # infinite costs
])
def test_stage_shapes_and_cost_extremes(ctx, t, prm):
    ex = synth.example(940, 33, 41)
    gen, job = run_pair([ex], 52, 40, seed=4, tuning=team(t), **prm)
    if prm.get("cauchy_dispersion", 1.0) == 0.0:
        assert np.array_equal(gen.coord, job.state()[1])  # NaN scores compare unequal
    else:
        assert_same(gen, job)


@pytest.mark.parametrize("t", [1, 8])
@pytest.mark.parametrize("px", [1, 5])
def test_fixed_batches_and_few_workgroups(ctx, t, px):
    # batches of 1 and 5 items (the first five find no resolved pixel), two workgroups
    ex = synth.example(950, 30, 30)
    sched = dict(px_per_batch=px, redo_shift=0, new_shift=0, max_batch=0, first_new_shift=0)
    gen, job = run_pair([ex], 36, 31, sched=sched, seed=2, tuning=team(t, flow_wgs=2))
    assert_same(gen, job)


def test_inpaint_and_mixed_teams(ctx):
    # teams change inside a stage (8, 4, then a wave per item), the hole's
    # neighbours come from the locked pixels, the items' mail and the state
    ex = synth.example(960, 160, 120)
    m = synth.ellipse_mask(961, 160, 120)
    gen, job = run_pair([ex], 160, 120, seed=6, inpaint_mask=m, inpaint_index=0, sample_kind=[2], sample_masks=[m],
                        tuning=dict(flow=1, ahead=1, prefetch_max=40, flow_head=16, team_waves=80))
    assert_same(gen, job)


def test_progress_images_are_the_batches_states(ctx):
    # the callback's images with and without dependency order are the same
    ex = synth.example(970, 64, 64)

    def images(flow):
        seen = []
        s = ts.Session.builder().add_example(ex).seed(9).output_size(ts.Dims(90, 70)).build().set_tuning(flow=flow)
        g = s.run(progress=lambda p: seen.append((p["total"], p["stage"], p["image"].copy())))
        return g, seen

    g1, s1 = images(1)
    g0, s0 = images(0)
    assert np.array_equal(g1.image, g0.image) and len(s1) == len(s0)
    for a, b in zip(s1, s0):
        assert a[0] == b[0] and a[1] == b[1] and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("t", [1, 8])
@pytest.mark.parametrize("ex,w,h,k,px", [
    (40, 23, 20, 12, 0),    # margins of one pixel
    (40, 61, 47, 50, 5),    # the first five pixels are resolved at random: no ghost copies
    (40, 19, 19, 30, 0),    # no margin: 5% of 19 is none
    (64, 330, 270, 50, 0),  # list, ring and table routes, partial edge tiles
])
def test_tiling_lists_by_rank(ctx, t, ex, w, h, k, px):
    sched = dict(ts.default_schedule(), px_per_batch=px)
    gen, job = run_pair([synth.example(980 + ex, ex, ex)], w, h, sched=sched, seed=w, nearest_neighbors=k,
                        tiling_mode=True, tuning=team(t))
    assert_same(gen, job)


@pytest.mark.parametrize("t", [2, 4, 8])
def test_offsets_far_beyond_the_examples(ctx, t):
    # the first items' neighbours lie several examples away, so that whole
    # members hold no valid candidate, and the maps differ in size
    exs = [synth.example(990, 9, 8), synth.example(991, 61, 57)]
    gen, job = run_pair(exs, 260, 230, seed=3, backtrack_stages=2, tuning=team(t))
    assert_same(gen, job)
