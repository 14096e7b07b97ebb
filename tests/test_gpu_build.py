"""What a job's build prepares on the device (pyramids of all images together,
style guides, the maps before the first stage) against the oracle, where its
kernels' rows, workgroups and groups end. Bit for bit."""
import numpy as np
import pytest

import tsgpu as ts
from oracle import refcpu as R
from tests.test_gpu_parity import assert_same, run_pair
from tsgpu import synth

pytestmark = pytest.mark.gpu


# rows just under, at and over a workgroup's 256 outputs; rows that share a
# workgroup; a single column of blocks; rows beyond one group's memory
@pytest.mark.parametrize("w,h,levels", [(255, 33, 4), (256, 40, 5), (257, 35, 5), (515, 301, 5), (16, 16, 5), (1, 1, 1),
                                        (2, 700, 2), (5003, 4801, 3)])
def test_pyramids(ctx, w, h, levels):
    img = synth.example(w + h, w, h)
    assert np.array_equal(ts.pyramid(img, levels, ctx), R.pyramid(img, levels))


@pytest.mark.parametrize("w,h,out_w,out_h", [(63, 41, 301, 259), (256, 64, 33, 47)])
def test_style_guides(ctx, w, h, out_w, out_h):
    exs = [synth.example(40 + i, w + 9 * i, h) for i in range(2)]
    gen, job = run_pair(exs, out_w, out_h, target_guide=synth.example(50, out_w, out_h), seed=3, backtrack_stages=2,
                        nearest_neighbors=9, random_sample_locations=7)
    assert_same(gen, job)


# points resolved before the stages: none left over, a list with moved
# entries, most of the list moved; the list on the device and on the host
@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("n", [1, 90, 700])
def test_random_init(ctx, n, flow):
    ex = synth.example(60, 33, 29)
    gen, job = run_pair([ex], 31, 25, seed=n, random_init=n, backtrack_stages=3, nearest_neighbors=12,
                        random_sample_locations=9, tuning=dict(flow=flow))
    assert_same(gen, job)


@pytest.mark.parametrize("flow", [0, 1])
@pytest.mark.parametrize("n", [None, 40])
def test_inpaint_start(ctx, n, flow):
    w, h = 77, 41
    mask = synth.ellipse_mask(5, w, h)
    kw = {} if n is None else dict(random_init=n)
    gen, job = run_pair([synth.example(70, w, h)], w, h, seed=2, inpaint_mask=mask, inpaint_index=0, sample_kind=[2],
                        sample_masks=[mask], backtrack_stages=3, tuning=dict(flow=flow), **kw)
    assert_same(gen, job)


# pixel counts that are not whole words of the mask; a mask larger than its example
@pytest.mark.parametrize("w,h", [(33, 29), (1, 50), (64, 33)])
def test_sample_masks(ctx, w, h):
    ex = synth.example(80, w, h)
    rng = np.random.default_rng(w)
    big = np.zeros((h + 3, w + 5, 4), np.uint8)
    big[:, :, 0] = (rng.random((h + 3, w + 5)) < 0.3) * rng.integers(1, 256, (h + 3, w + 5))
    mask = np.ascontiguousarray(big[:h, :w])
    kw = dict(seed=6, sample_kind=[2], backtrack_stages=0, nearest_neighbors=9, random_sample_locations=7)
    gen, job = run_pair([ex], 40, 31, sample_masks=[mask], **kw)
    assert_same(gen, job)
    b = ts.Session.builder().seed(6).backtrack_stages(0).nearest_neighbors(9).random_sample_locations(7)
    got = b.add_example(ts.Example(ex).set_sample_method(big)).output_size(ts.Dims(40, 31)).build().run()
    assert np.array_equal(got.image, gen.image) and np.array_equal(got.coord, gen.coord)
