"""The persistent traversal at its edges: ray counts around a wave, a chunk and
a block, trees whose nodes hit many primitives at once for every lane (the
ring of waiting ray/primitive pairs fills several times per step), coincident
primitives (equal t: the lower id wins), one bounce only, and shadow rays in a
launch of their own.  Every render must equal the oracle's: the same float
operations per path, in the same order, so radiance within 1e-3 of every pixel
(as the other parity tests; 99.99% of pixels bit-identical)."""
import numpy as np
import pytest

import oracle
import pupiloptixlab_amd as pt

pytestmark = pytest.mark.gpu

STACK = """<scene version="3.0.0">
  <integrator type="path"><integer name="max_depth" value="{depth}"/></integrator>
  <sensor type="perspective"><float name="fov" value="40"/>
    <transform name="to_world"><lookat origin="0.1, 0.2, 4" target="0, 0, 0" up="0, 1, 0"/></transform>
    <film type="hdrfilm"><integer name="width" value="{w}"/><integer name="height" value="{h}"/></film>
  </sensor>
  {shapes}
  <shape type="rectangle"><transform name="to_world"><scale value="0.5"/><translate value="0, 0, 3.5"/></transform>
    <bsdf type="diffuse"/><emitter type="area"><rgb name="radiance" value="5, 4, 3"/></emitter></shape>
  <emitter type="constant"><rgb name="radiance" value="0.3"/></emitter>
</scene>"""


def stack_scene(tmp_path, w, h, depth=4, sheets=60, sphere=False):
    """Sheets one behind the other, every third one coincident with the one before."""
    shapes = []
    for k in range(sheets):
        z = -0.01 * (k - (1 if k % 3 == 2 else 0))
        shapes.append(f"""<shape type="rectangle"><transform name="to_world"><translate value="0, 0, {z}"/></transform>
            <bsdf type="twosided"><bsdf type="diffuse"><rgb name="reflectance" value="{0.2 + 0.01 * k}, 0.5, 0.4"/>
            </bsdf></bsdf></shape>""")
    if sphere:
        shapes.append('<shape type="sphere"><transform name="to_world"><scale value="0.4"/></transform>'
                      '<bsdf type="diffuse"/></shape>')
    p = tmp_path / "stack.xml"
    p.write_text(STACK.format(w=w, h=h, depth=depth, shapes="\n".join(shapes)))
    return pt.HostScene.load_xml(str(p))


def check(tracer, scene, spp, **kw):
    tracer.set_scene(scene)
    tracer.build_bvh()
    tracer.render(spp=spp, **kw)
    got, prim = tracer.read(pt.BUF_ACCUM), tracer.read(pt.BUF_PRIM_ID)
    ref = oracle.render(scene.desc, spp=spp, **{k: v for k, v in kw.items() if k == "max_depth"})
    g, r = got[..., :3].astype(np.float64), ref["accum"][..., :3].astype(np.float64)
    assert np.all(np.abs(g - r) <= 1e-3 * np.abs(r) + 1e-6)
    assert np.mean(np.all(g == r, axis=-1)) >= 0.9999
    assert np.array_equal(prim, ref["prim"])


@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (63, 1, 1), (64, 1, 1), (65, 1, 1), (16, 16, 1), (257, 3, 2),
                                     (96, 80, 3)])
@pytest.mark.parametrize("one_chain", [False, True])
def test_many_primitives_per_node_and_ties(tracer, tmp_path, w, h, spp, one_chain):
    print(f"case: stacked sheets {w}x{h} {spp} spp one_chain={one_chain}", flush=True)
    check(tracer, stack_scene(tmp_path, w, h), spp, one_chain=one_chain)


@pytest.mark.parametrize("depth", [1, 2, 3])
def test_first_bounces(tracer, tmp_path, depth):
    print(f"case: stacked sheets with a sphere 70x50 depth {depth}", flush=True)
    check(tracer, stack_scene(tmp_path, 70, 50, sphere=True), 2, max_depth=depth)


def test_more_rays_than_the_grid(tracer):
    """1.6 M camera rays: waves refill from the cursor; against the same frames one by one."""
    print("case: terrain 640x512 5 frames, one launch vs one launch per frame", flush=True)
    scene = pt.HostScene.generate(pt.SCENE_TERRAIN, seed=5, width=640, height=512, grid=96, spheres=24)
    tracer.set_scene(scene)
    tracer.build_bvh()
    tracer.render(spp=5)
    a = tracer.read(pt.BUF_ACCUM)
    tracer.reset()
    tracer.render(spp=5, spp_per_launch=1, one_chain=True)
    assert np.array_equal(a, tracer.read(pt.BUF_ACCUM))


@pytest.mark.parametrize("spheres", [0, 24])
def test_counts_are_the_rays_own(tracer, spheres):
    """Node visits and primitive tests of the same frames do not depend on launch width, on which rays share a
    launch or on the run, and counting does not change the image."""
    print(f"case: counting, terrain 322x181 with {spheres} spheres, 4 frames", flush=True)
    scene = pt.HostScene.generate(pt.SCENE_TERRAIN, seed=6, width=322, height=181, grid=128, spheres=spheres)
    tracer.set_scene(scene)
    tracer.build_bvh()
    tracer.render(spp=4)
    image = tracer.read(pt.BUF_ACCUM)
    keys = ("rays_extension", "rays_shadow", "node_visits", "tri_tests", "shadow_node_visits", "shadow_tri_tests")
    counts = []
    tracer.set_counting(True)
    try:
        for per, one in ((4, False), (4, False), (4, True), (1, False), (3, True)):
            tracer.reset()
            before = tracer.stats()
            tracer.render(spp=4, spp_per_launch=per, one_chain=one)
            after = tracer.stats()
            counts.append({k: after[k] - before[k] for k in keys})
            assert np.array_equal(image, tracer.read(pt.BUF_ACCUM))
    finally:
        tracer.set_counting(False)
    assert all(c == counts[0] for c in counts) and min(counts[0].values()) > 0


def test_times_of_launches_that_take_both_kinds_of_rays(tracer):
    """Timed renders, direct batches too: a launch with extension and shadow rays counts for both kinds."""
    print("case: timed renders of 2 launches at depth 6, shared and separate shadow launches, and a batch", flush=True)
    scene = pt.HostScene.generate(pt.SCENE_CORNELL, width=160, height=120)
    tracer.set_scene(scene)
    tracer.build_bvh()
    keys = ("ms_trace", "ms_shadow", "launches_trace", "launches_shadow")

    def timed(call):
        before = tracer.stats()
        call()
        after = tracer.stats()
        return [after[k] - before[k] for k in keys]

    for one in (False, True):
        ms_trace, ms_shadow, n_trace, n_shadow = timed(
            lambda: tracer.render(spp=4, max_depth=6, spp_per_launch=2, timing=True, one_chain=one))
        assert (n_trace, n_shadow) == (2 * 6, 2 * 5)
        assert 0.0 < ms_shadow and 0.0 < ms_trace
        assert one or ms_shadow < ms_trace  # a part of the same launches
    tracer.batch_clear()
    tracer.batch_add_view(scene, 2)
    ms_trace, ms_shadow, n_trace, n_shadow = timed(lambda: tracer.batch_render(graph=False, timing=True))
    tracer.batch_clear()
    depth = scene.desc.max_depth
    assert n_trace % depth == 0 and n_shadow * depth == n_trace * (depth - 1) and 0.0 < ms_shadow < ms_trace
