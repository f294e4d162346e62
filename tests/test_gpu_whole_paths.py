"""Small path-tracer batches, traced in one launch, equal the wavefront queues bit for bit.

A batch of up to 1024 paths per CU (262,144 on 256 CUs; 65,536 for plain frames in a shallow tree) runs each path in
registers, 64 paths a wave or, in small batches and deep trees, 8 to 32 with several lanes per ray. Timing a frame's
stages keeps the queues; both add the same terms to a path in the same order.
"""
import numpy as np
import pytest

import cupbr_amd as cb
from cupbr_amd import scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "cornell": lambda: scenes.cornell_box(),
    "mixed": lambda: scenes.mixed_primitives(env=True),
    "boxes": lambda: scenes.million_triangles(n_spheres=2, subdiv=4, n_boxes=300),  # a deep tree
}


def _frame(scene, ca, w, h, spp, depth, queues, rr=False, rng=0, cache=None):
    r = cb.PBRenderer(cb.RenderingMethod.PATHTRACER)
    r.set_output_size(w, h)
    r.register_scene(scene)
    r.set_max_trace_depth(depth)
    r.set_russian_roulette(rr)
    r.set_rng(rng)
    if cache is not None:
        r.set_radiance_cache(cache, training_paths=w * h // 4, train_steps=0)
    r.set_profiling(queues)
    r.render(cb.Camera.look_at(ca["eye"], ca["target"], ca["up"], ca["vfov"], w, h), spp)
    st = r.stats()
    return r.get_output_image(), {k: st[k] for k in ("extension_rays", "shadow_rays", "cache_queries", "cache_training_rows")}


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("w,h,spp,depth,rr,rng", [
    (1, 1, 1, 5, False, 0), (7, 5, 1, 1, False, 0), (13, 11, 3, 9, True, 0),
    (128, 128, 1, 4, False, 1),   # the last batch of 8 paths a wave in a shallow tree
    (113, 145, 1, 6, True, 0),    # one more: 64 a wave
    (256, 257, 1, 5, False, 0), (512, 512, 1, 3, True, 1),  # the largest batch
    (512, 513, 1, 3, False, 0),   # queues
])
def test_whole_paths_equal_queues(name, w, h, spp, depth, rr, rng):
    desc, ca = SCENES[name]()
    scene = cb.Scene.from_desc(desc)
    got, n_got = _frame(scene, ca, w, h, spp, depth, False, rr, rng)
    want, n_want = _frame(scene, ca, w, h, spp, depth, True, rr, rng)
    print(f"{name} {w}x{h} {spp} spp depth {depth}: {n_got}", flush=True)
    assert n_got == n_want and n_got["extension_rays"] >= w * h * spp
    assert np.array_equal(got, want)


@pytest.mark.parametrize("name", ["cornell", "mixed"])
@pytest.mark.parametrize("w,h,spp,depth", [
    (256, 256, 1, 2), (128, 64, 8, 5),    # the last whole paths of more bounces than one in a shallow tree
    (331, 199, 1, 2),                     # queues
    (256, 192, 1, 1), (223, 221, 1, 1),   # the last of one bounce, and queues
])
def test_limits_of_plain_frames_in_shallow_trees(name, w, h, spp, depth):
    test_whole_paths_equal_queues(name, w, h, spp, depth, False, 0)


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("w,h", [(37, 29), (256, 256), (300, 299)])
def test_cached_whole_paths_equal_queues(name, w, h):
    """The same with a radiance cache (without training steps, so that both frames ask the same weights)."""
    desc, ca = SCENES[name]()
    scene = cb.Scene.from_desc(desc)
    cache = cb.RadianceCache((-3, -3, -3), (3, 3, 3), seed=3)
    got, n_got = _frame(scene, ca, w, h, 2, 6, False, cache=cache)
    want, n_want = _frame(scene, ca, w, h, 2, 6, True, cache=cache)
    assert n_got == n_want and n_got["cache_queries"] > 0 and n_got["cache_training_rows"] > 0
    assert np.array_equal(got, want)


@pytest.mark.parametrize("name,w,h", [("cornell", 21, 13), ("cornell", 200, 161), ("boxes", 96, 64), ("cornell", 512, 512)])
def test_whole_paths_leave_the_rows_of_the_queues(name, w, h):
    """Every path a training path: the rows, gathered from one part per XCD, are as many as the queues' and the
    Adam step on a million draws of them goes the same way. A weight's first step is lr against the sign of its
    gradient, whose sampling error is 1e-3 of the rows' spread. Of the last size's rows 2^18 are kept, which ones
    is up to their order (the queues keep the first bounces')."""
    desc, ca = SCENES[name]()
    scene = cb.Scene.from_desc(desc)
    cam = cb.Camera.look_at(ca["eye"], ca["target"], ca["up"], ca["vfov"], w, h)
    steps, rows, images = [], [], []
    for queues in (False, True):
        cache = cb.RadianceCache((-3, -3, -3), (3, 3, 3), seed=3)
        w0 = cache.get_weights()
        r = cb.PBRenderer(cb.RenderingMethod.PATHTRACER)
        r.set_output_size(w, h)
        r.register_scene(scene)
        r.set_max_trace_depth(6)
        r.set_radiance_cache(cache, training_paths=w * h, train_steps=1, batch=1 << 20, learning_rate=1e-3)
        r.set_profiling(queues)
        r.render(cam, 1)
        rows.append(r.stats()["cache_training_rows"])
        images.append(r.get_output_image())
        steps.append((cache.get_weights() - w0).astype(np.float64))
    print(f"{name} {w}x{h}: {rows} rows", flush=True)
    assert rows[0] == rows[1] > 0 and (rows[0] == 1 << 18) == (w == 512)
    assert np.array_equal(images[0], images[1])
    assert np.isfinite(steps[0]).all()
    a, b = steps
    assert rows[0] == 1 << 18 or np.dot(a, b) >= 0.95 * np.linalg.norm(a) * np.linalg.norm(b)


def _cached(scene, cam, w, h, calls, depth=6, weights=None, **kw):
    """(image, counts, weights afterwards) of a cached render in calls of so many frames"""
    cache = cb.RadianceCache((-3, -3, -3), (3, 3, 3), seed=3)
    if weights is not None:
        cache.set_weights(weights)
    r = cb.PBRenderer(cb.RenderingMethod.PATHTRACER)
    r.set_output_size(w, h)
    r.register_scene(scene)
    r.set_max_trace_depth(depth)
    r.set_radiance_cache(cache, **kw)
    counts = np.zeros(4, np.int64)
    for spp in calls:
        r.render(cam, spp)
        st = r.stats()
        counts += [st[k] for k in ("extension_rays", "shadow_rays", "cache_queries", "cache_training_rows")]
    return r.get_output_image(), counts, cache.get_weights()


@pytest.mark.parametrize("name", ["cornell", "mixed"])
@pytest.mark.parametrize("training", [0, 8])
def test_large_cached_batches_equal_smaller_ones(name, training):
    """A batch of 2^20 paths asks the cache for the first queries on a second stream, the rest (behind mirrors and
    glass) after the last bounce; two calls of half as many paths ask once. Their frames are the same."""
    w, h = 1024, 600
    desc, ca = SCENES[name]()
    scene = cb.Scene.from_desc(desc)
    cam = cb.Camera.look_at(ca["eye"], ca["target"], ca["up"], ca["vfov"], w, h)
    kw = dict(training_paths=w * h * training // 64, train_steps=0)
    a, n_a, _ = _cached(scene, cam, w, h, [2], **kw)
    b, n_b, _ = _cached(scene, cam, w, h, [1, 1], **kw)
    assert n_a[2] > 0 and (n_a[3] > 0) == (training > 0)
    assert np.array_equal(n_a, n_b) and np.array_equal(a, b)


def test_large_cached_batches_keep_the_estimator():
    """The same size with a zero cache (every path ends at its second vertex) and with training paths alone."""
    w, h = 1024, 600
    desc, ca = SCENES["cornell"]()
    scene = cb.Scene.from_desc(desc)
    cam = cb.Camera.look_at(ca["eye"], ca["target"], ca["up"], ca["vfov"], w, h)
    zero, counts, _ = _cached(scene, cam, w, h, [2], weights=np.zeros(cb.NRC_PARAMS, np.float32), training_paths=0,
                              train_steps=0)
    assert counts[2] > 0 and np.array_equal(zero, _frame(scene, ca, w, h, 2, 1, False)[0])
    w0 = cb.RadianceCache((-3, -3, -3), (3, 3, 3), seed=3).get_weights()
    full, counts, trained = _cached(scene, cam, w, h, [2], training_paths=w * h, train_steps=2, batch=4096)
    assert counts[2] == 0 and counts[3] > 0 and np.array_equal(full, _frame(scene, ca, w, h, 2, 6, False)[0])
    assert np.isfinite(trained).all() and not np.array_equal(trained, w0)
