"""Network queries in spatial order (queues of 2^16 slots and more) against
queries in queue order (smaller queues): each query's outputs go to its own
slot, so the same frames in wide and in narrow launches give the same image,
bit for bit, with one hash grid and with one per batch view."""
import ctypes as C

import numpy as np
import pytest

import pupiloptixlab_amd as pt

pytestmark = pytest.mark.gpu


def params(seed, grids=1, log2_t=14):
    rng = np.random.default_rng(seed)
    shape = (16, 1 << log2_t, 2) if grids == 1 else (grids, 16, 1 << log2_t, 2)
    dims = [32, 64, 64, 64, 41]
    w = np.zeros((4, 64, 64), np.float32)
    for l in range(4):
        w[l, :dims[l], :dims[l + 1]] = rng.normal(0, 1.2 / np.sqrt(dims[l]), (dims[l], dims[l + 1]))
    return rng.normal(0, 0.3, shape).astype(np.float32), w


@pytest.mark.parametrize("kind,w,h,frames", [(pt.SCENE_DOOR_ROOM, 257, 33, 9), (pt.SCENE_TERRAIN, 256, 128, 2)])
def test_wide_and_narrow_launches(tracer, kind, w, h, frames):
    print(f"case: guided {w}x{h}, {frames} frames in one launch (sorted) and one by one", flush=True)
    assert w * h < 1 << 16 <= w * h * frames
    scene = pt.HostScene.generate(kind, seed=3, width=w, height=h, grid=64)
    tracer.set_scene(scene)
    tracer.build_bvh()
    tracer.guide_enable(log2_table=14)
    tracer.guide_set_params(*params(1))
    out = []
    for per in (frames, 1):
        tracer.reset()
        q0 = tracer.stats()["guide_queries"]
        tracer.render(spp=frames, mis_mode=pt.MIS_CONSISTENT, guide=True, spp_per_launch=per)
        out.append((tracer.read(pt.BUF_ACCUM), tracer.stats()["guide_queries"] - q0))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1] > 0
    tracer.guide_disable()


@pytest.mark.parametrize("views", [1, 3, 5])
def test_batch_grids(tracer, views):
    print(f"case: guided batch of {views} views, wide (sorted) and narrow launches", flush=True)
    tracer.batch_clear()
    for v in range(views):
        scene = pt.HostScene.generate(pt.SCENE_CORNELL_VARIANT, seed=v + 1, triangles=2000, width=190, height=97)
        tracer.batch_add_view(scene, 5)
    tracer.guide_enable_batch(log2_table=14)
    tracer.guide_set_params(*params(2, views))
    out = []
    for paths, graph in ((1 << 18, True), (20000, False)):
        tracer.batch_reset()
        tracer.batch_render(mis_mode=pt.MIS_CONSISTENT, guide=True, paths_per_launch=paths, graph=graph)
        out.append([tracer.batch_read(v) for v in range(views)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    tracer.guide_disable()
    tracer.batch_clear()


def test_first_sort_of_a_context():
    """The histogram's first clear is ordered before the first sort, whatever
    the memory held: contexts made where others left their queues, sorted
    inference first thing."""
    scene = pt.HostScene.generate(pt.SCENE_DOOR_ROOM, seed=3, width=257, height=160)
    want = None
    for k, per in enumerate((1, 2, 2, 2)):
        print(f"case: context {k}, {per} frames per launch at once", flush=True)
        with pt.PathTracer(0) as t:
            t.set_scene(scene)
            t.build_bvh()
            t.guide_enable(log2_table=14)
            t.guide_set_params(*params(1))
            t.render(spp=2, mis_mode=pt.MIS_CONSISTENT, guide=True, spp_per_launch=per)
            got = t.read(pt.BUF_ACCUM)
        want = got if want is None else want
        assert np.array_equal(got, want)


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert pt.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_no_sorting_buffers_for_what_is_not_sorted():
    """A guided batch with queues for 2^22 paths whose launches are narrow holds 96 bytes per slot for the network's
    outputs and no more."""
    slots = 1 << 22
    print("case: guided batch, launches of 12 K paths in queues of 4 M", flush=True)
    with pt.PathTracer(0) as t:
        t.batch_add_view(pt.HostScene.generate(pt.SCENE_CORNELL_VARIANT, seed=1, triangles=2000, width=128, height=96), 1)
        t.guide_enable_batch(log2_table=14)
        t.guide_set_params(*params(2))
        kw = {"mis_mode": pt.MIS_CONSISTENT, "paths_per_launch": slots, "graph": False}
        t.batch_render(**kw)
        before = free_bytes()
        t.batch_render(guide=True, **kw)
        assert before - free_bytes() < 96 * slots + (32 << 20)
