"""Workloads of the framework's public entry points, for timing and comparing.

Each case is one thing that a program using tsgpu does, from decoded images on
the host to the finished maps on the host: SessionBuilder.build (upload,
pyramids, initial state) and Session.run (random init, every backtracking
stage, download), Batch and Server for many syntheses, and
CoordinateTransform.apply. Images go in and come out as host arrays by the
API's nature, so a pass is the whole call.

Inputs are the seeded images of tsgpu.synth, the distributions of the
repository's benchmark and tests. `k`, `m` are nearest_neighbors and
random_sample_locations. Run from the repository's root.
"""
import math
import os
import sys

import numpy as np

_PKG = os.path.abspath("texture-synthesis_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tsgpu as ts  # noqa: E402
from tsgpu import serve, synth  # noqa: E402

#: Output pixels a drawn case may have, by kind, so that none costs more than
#: the largest listed case (2048^2 from one example).
MOST_PX = {"texture": 2048 * 2048, "multi": 1400 * 1400, "guided": 1024 * 1024, "style": 1024 * 1024,
           "inpaint": 1400 * 1400, "tiling": 640 * 640, "transform": 2048 * 2048}
KINDS = ("texture", "texture", "multi", "guided", "style", "inpaint", "tiling", "batch", "serve", "transform")


def listed():
    return [
        # a thumbnail or a tile: every launch is small, so launches and latency count
        dict(name="texture_64", kind="texture", ex_w=48, ex_h=48, w=64, h=64, k=50, m=50, stages=5),
        # the reference's own small benchmark case
        dict(name="texture_256", kind="texture", ex_w=128, ex_h=128, w=256, h=256, k=50, m=50, stages=5),
        # the headline: a 1024^2 texture from a 512^2 example at the defaults
        dict(name="texture_1024", kind="texture", ex_w=512, ex_h=512, w=1024, h=1024, k=50, m=50, stages=5),
        # a large texture
        dict(name="texture_2048", kind="texture", ex_w=512, ex_h=512, w=2048, h=2048, k=50, m=50, stages=5),
        # several examples of odd sizes, one of them masked, random seeding, at the default 500-pixel
        # output cut to a ragged height; the coordinate maps are taken too (a transform is saved)
        dict(name="multi_500x333", kind="multi", ex_w=203, ex_h=151, n_ex=3, w=500, h=333, k=20, m=50, stages=5),
        # guided synthesis: four examples with guide maps and a target guide
        dict(name="guided_1024", kind="guided", ex_w=300, ex_h=300, n_ex=4, w=1024, h=1024, k=50, m=50, stages=5),
        # style transfer: a target image as guide, the example's guide derived from it
        dict(name="style_640x427", kind="style", ex_w=256, ex_h=256, w=640, h=427, k=50, m=50, stages=5),
        # filling 20-40% of a picture of odd size from an example resized to it
        dict(name="inpaint_731x557", kind="inpaint", ex_w=256, ex_h=256, w=731, h=557, k=50, m=50, stages=5),
        # a texture that tiles, for a game's material
        dict(name="tiling_401x300", kind="tiling", ex_w=200, ex_h=200, w=401, h=300, k=50, m=50, stages=5),
        # an offline batch: 48 syntheses together on the work-queue engine
        dict(name="batch_48", kind="batch", n=48, k=50, m=50, stages=5),
        # a burst of requests at the serving loop, plain and inpainting, small and large
        dict(name="serve_16", kind="serve", n=16, k=50, m=50, stages=5),
        # a saved transform applied to another picture of the example's size
        dict(name="transform_1024", kind="transform", ex_w=512, ex_h=512, n_ex=2, w=1024, h=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    if kind == "batch":
        return dict(kind=kind, n=rng.randint(9, 47), k=rng.choice((20, 50)), m=rng.choice((20, 35, 50)), stages=5)
    if kind == "serve":
        return dict(kind=kind, n=rng.randint(2, 15), k=rng.choice((20, 50)), m=rng.choice((20, 35, 50)), stages=5)
    most = math.sqrt(MOST_PX[kind])
    side = math.exp(rng.uniform(math.log(64.0), math.log(most / 1.15)))
    aspect = math.exp(rng.uniform(-0.25, 0.25))
    case = dict(kind=kind, ex_w=_log(rng, 48, 512), ex_h=_log(rng, 48, 512), w=max(48, int(side * aspect)),
                h=max(48, int(side / aspect)))
    if kind in ("multi", "guided", "transform"):
        case["n_ex"] = rng.randint(2, 4)
    if kind != "transform":
        case.update(k=rng.choice((20, 50, 50)), m=rng.choice((20, 50, 50)), stages=rng.choice((3, 5, 5)))
    return case


def _batch_specs(n):
    """(example side, output side) pairs of a batch: the benchmark's mix, its
    512 example and 1024 output sizes left out."""
    return [((64, 128, 256)[i // 3 % 3], (128, 256, 512)[i % 3]) for i in range(n)]


def _serve_specs(n):
    """(output side, inpainting) pairs of a burst: sides spread evenly in
    their logarithm over 128..1024, from 256^2 examples, in mixed order, 30%
    inpainting."""
    order = sorted(range(n), key=lambda i: (i * 0.618034) % 1.0)
    return [(int(128.0 * 8.0 ** ((i + 0.5) / n)), i % 10 % 3 == 1) for i in order]


def _builder(case, seed):
    b = ts.Session.builder().seed(seed).nearest_neighbors(case["k"]).random_sample_locations(case["m"])
    return b.backtrack_stages(case["stages"])


def _request(case, seed, side, inpaint):
    b = _builder(case, seed)
    ex = synth.example(seed, 256, 256)
    if inpaint:
        m = synth.ellipse_mask(seed, side, side)
        return b.inpaint_example(m, ts.Example(ex).set_sample_method(m), ts.Dims.square(side))
    return b.add_example(ex).output_size(ts.Dims.square(side))


def prepare(case, seed):
    """The decoded images and the builder (or server, batch, transform) that a
    program holds before the call."""
    kind = case["kind"]
    ts.Context.default()
    if kind == "batch":
        bs = [_builder(case, seed + j).add_example(synth.example(seed + j, e, e)).output_size(ts.Dims.square(o))
              for j, (e, o) in enumerate(_batch_specs(case["n"]))]
        return dict(kind=kind, builders=bs, batch=ts.Batch(max_active=256))
    if kind == "serve":
        bs = [_request(case, seed + i, s, p) for i, (s, p) in enumerate(_serve_specs(case["n"]))]
        return dict(kind=kind, builders=bs, server=serve.Server(hbm_budget=4 << 30))
    w, h, ew, eh = case["w"], case["h"], case["ex_w"], case["ex_h"]
    if kind == "transform":
        rng = np.random.default_rng(seed)
        n = case["n_ex"]
        # patches of consecutive source pixels, as a synthesis leaves them
        gx, gy = (w + 15) // 16, (h + 15) // 16
        ox, oy = rng.integers(0, ew, (gy, gx)), rng.integers(0, eh, (gy, gx))
        om = rng.integers(0, n, (gy, gx))
        up = [np.repeat(np.repeat(a, 16, 0), 16, 1)[:h, :w] for a in (ox, oy, om)]
        xs, ys = np.meshgrid(np.arange(w), np.arange(h))
        buf = np.stack([(up[0] + xs) % ew, (up[1] + ys) % eh, up[2]], -1).astype(np.uint32).reshape(-1)
        ct = ts.CoordinateTransform(buf, ts.Dims(w, h), [ts.Dims(ew, eh)] * n)
        return dict(kind=kind, transform=ct, sources=[synth.example(seed + i, ew, eh) for i in range(n)])
    b = _builder(case, seed)
    if kind == "texture":
        b.add_example(synth.example(seed, ew, eh)).output_size(ts.Dims(w, h))
    elif kind == "multi":
        for i in range(case["n_ex"]):
            # odd sizes, each its own
            e = ts.Example(synth.example(seed + i, ew + 8 * i, eh + 5 * i))
            if i == 1:
                e.set_sample_method(synth.ellipse_mask(seed + i, ew + 8 * i, eh + 5 * i))
            b.add_example(e)
        b.random_init(10).output_size(ts.Dims(w, h))
    elif kind == "guided":
        for i in range(case["n_ex"]):
            b.add_example(ts.Example(synth.example(seed + i, ew, eh)).with_guide(synth.blobs(seed + 50 + i, ew, eh)))
        b.load_target_guide(synth.blobs(seed + 99, w, h)).random_init(10).output_size(ts.Dims(w, h))
    elif kind == "style":
        b.add_example(synth.example(seed, ew, eh)).load_target_guide(synth.example(seed + 1, w, h))
        b.output_size(ts.Dims(w, h))
    elif kind == "inpaint":
        m = synth.ellipse_mask(seed, w, h)
        b.inpaint_example(m, ts.Example(synth.example(seed, ew, eh)).set_sample_method(m), ts.Dims(w, h))
    elif kind == "tiling":
        b.add_example(synth.example(seed, ew, eh)).tiling_mode(True).output_size(ts.Dims(w, h))
    else:
        raise ValueError(f"unknown kind {kind}")
    return dict(kind=kind, builder=b)


def _maps(g):
    return dict(image=g.image, resolved=g.resolved_flat, score=g.resolved_score)


def run(state):
    kind = state["kind"]
    if kind == "transform":
        return dict(image=state["transform"].apply(state["sources"]))
    if kind == "batch":
        batch = state["batch"]
        tickets = [batch.submit(b.build()) for b in state["builders"]]
        batch.run_all()
        return [batch.take(t).image for t in tickets]
    if kind == "serve":
        server = state["server"]
        for b in state["builders"]:
            server.submit(b)
        done = sorted(server.drain(), key=lambda f: f.rid)
        if any(f.error is not None for f in done):
            raise RuntimeError(next(str(f.error) for f in done if f.error is not None))
        return [f.result.image for f in done]
    g = state["builder"].build().run()
    out = _maps(g)
    if kind == "multi":
        out["coord"], out["ids"] = g.coord, g.ids
    return out


#: One output pixel's maps: the 16-byte record, its place in the resolved
#: order and its score.
_OUT_BYTES = 24


def _synthesis_work(case, w, h, in_px, guided=False):
    """A synthesis reads its images once and writes its maps once. Its
    operations: over the stages every pixel is resolved (1 - p^(P+1)) / (1 - p)
    times (p = 0.5), and each resolve compares k neighbours of k + m
    candidates, of which exact pruning needs about 15%: four channel
    differences, table terms and adds, and a weighting (14 operations; with
    guides twice the channels)."""
    n = w * h
    resolves = n * (2.0 - 0.5 ** case["stages"])
    terms = 0.15 * case["k"] * (case["k"] + case["m"])
    return {"bytes": 4 * in_px + _OUT_BYTES * n, "flops": resolves * terms * (26 if guided else 14)}


def work(case):
    kind = case["kind"]
    if kind == "transform":
        n = case["w"] * case["h"]
        return {"bytes": 16 * n + 4 * case["n_ex"] * case["ex_w"] * case["ex_h"], "flops": 0}
    if kind in ("batch", "serve"):
        if kind == "batch":
            parts = [_synthesis_work(case, o, o, e * e) for e, o in _batch_specs(case["n"])]
        else:
            parts = []
            for s, p in _serve_specs(case["n"]):
                part = _synthesis_work(case, s, s, 256 * 256 + (s * s if p else 0))
                part["flops"] *= 0.3 if p else 1.0  # the holes alone are resolved
                parts.append(part)
        return {q: sum(p[q] for p in parts) for q in ("bytes", "flops")}
    n_ex = case.get("n_ex", 1)
    px = n_ex * case["ex_w"] * case["ex_h"]
    n = case["w"] * case["h"]
    if kind == "guided":
        px = 2 * px + n
    elif kind in ("style", "inpaint"):
        px += n  # the target guide, or the mask
    work_ = _synthesis_work(case, case["w"], case["h"], px, guided=kind in ("guided", "style"))
    if kind == "inpaint":
        work_["flops"] *= 0.3  # the holes alone are resolved
    return work_


def exact(case, seed):
    """Syntheses have no 64-bit value beside the search itself (their maps are
    indices and bytes, and the scores follow the search); a transform's image
    is its gather."""
    if case["kind"] != "transform":
        return None
    state = prepare(case, seed)
    c = state["transform"].buffer.reshape(-1, 3).astype(np.int64)
    srcs = np.stack(state["sources"])
    return dict(image=srcs[c[:, 2], c[:, 1], c[:, 0]].reshape(case["h"], case["w"], 4))
