"""Edges of the wavefront queues: how rays are handed out must not show in the images."""
import numpy as np
import pytest

import cupbr_amd as cb
from cupbr_amd import scenes

pytestmark = pytest.mark.gpu


def _image(scene, ca, w, h, spp, method, depth, counting):
    r = cb.PBRenderer(method)
    r.set_output_size(w, h)
    r.register_scene(scene)
    r.set_max_trace_depth(depth)
    r.set_traversal_counting(counting)
    r.render(cb.Camera.look_at(ca["eye"], ca["target"], ca["up"], ca["vfov"], w, h), spp)
    return r.get_output_image(), r.stats()["refill_launches"]


@pytest.mark.parametrize("w,h,spp", [(641, 479, 2), (512, 512, 3), (1025, 769, 1), (331, 317, 9)])
def test_handed_out_rays_equal_dealt_chunks(w, h, spp):
    """Launches of at least one ray per lane of the persistent grid (524,288 rays on 256 CUs) hand each
    XCD's rays out in pieces, the others and the visit-counting mode deal 64-ray chunks. These sizes
    leave whole and partial granules, XCDs with fewer rays than their first pieces, and launches on
    both sides of the limit; each path's image is the same sum whoever traces its rays."""
    desc, ca = scenes.mixed_primitives(env=True)
    scene = cb.Scene.from_desc(desc)
    got, refills = _image(scene, ca, w, h, spp, cb.RenderingMethod.PATHTRACER, 6, False)
    want, none = _image(scene, ca, w, h, spp, cb.RenderingMethod.PATHTRACER, 6, True)
    assert refills > 0 and none == 0
    assert np.isfinite(got).all() and float(got.mean()) > 0
    assert np.array_equal(got, want)
