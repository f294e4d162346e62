"""Scenes whose tree is about as deep as the builder makes it (32 levels, 97 stack entries per ray).

Sizes in geometric progression leave a chain of ever smaller boxes. Walked by a group of lanes per ray, such a tree
brings the stack to where a step takes one entry instead of several, and per lane it spills the stack.
"""
import numpy as np
import pytest

import cupbr_amd as cb
import oracle
from cupbr_amd import scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _chain():
    b = scenes.SceneBuilder()
    m = scenes.material(scenes.LAMBERT, albedo_d=(0.7, 0.6, 0.5))
    for i in range(281):
        c = 1e-12 * 1.2228 ** i
        b.sphere((c, 0.5 * c, -c), 0.5514 * c, m)
    b.point_light((0.0, 5.0, 0.0), (40.0, 40.0, 40.0))
    return b.desc()


def _rays(n, seed):
    """From near the chain's point, along it: into the spheres and past them through the corners of their boxes."""
    rng = np.random.default_rng(seed)
    size = 10.0 ** rng.uniform(-13, 8, (n, 1))
    o = rng.normal(0, 0.2, (n, 3)) * size
    d = np.array([1.0, 0.5, -1.0]) + rng.uniform(-0.6, 0.6, (n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, d], 1).astype(np.float32), (10.0 ** rng.uniform(-12, 12, n)).astype(np.float32)


def test_queries_in_a_deep_tree():
    desc = _chain()
    S = cb.Scene.from_desc(desc)
    assert S.bvh_stats()["stack_entries"] > 90
    rays, dist = _rays(170_000, 3)
    rays_d, dist_d = torch.from_numpy(rays).cuda(), torch.from_numpy(dist).cuda()
    whole = [x.cpu().numpy() for x in (*S.trace_closest(rays_d), S.trace_visibility(rays_d, dist_d))]
    assert 0.1 < np.mean(whole[0] >= 0) < 0.9 and 0.1 < np.mean(whole[3]) < 0.9
    for count in (63, 8192, 32768, 163_840):  # 64, 64, 32 and 16 lanes a ray
        print(f"{count} rays", flush=True)
        part = [x.cpu().numpy() for x in (*S.trace_closest(rays_d[:count].contiguous()),
                                          S.trace_visibility(rays_d[:count].contiguous(), dist_d[:count].contiguous()))]
        for a, b in zip(whole, part):
            assert np.array_equal(a[:count].view(np.uint8), b.view(np.uint8))
    ref = oracle.OracleScene(desc, precisions=(32,))
    for a, b in zip(ref.trace(rays[:4096], precision=32, mode=0), whole):
        assert np.array_equal(a, b[:4096])
    assert np.array_equal(ref.visibility(rays[:4096], dist[:4096], precision=32, mode=0), whole[3][:4096])


@pytest.mark.parametrize("w,h", [(7, 5), (64, 48), (256, 200)])
def test_frames_in_a_deep_tree(w, h):
    """Whole paths, whose waves' last rays take 8 lanes each, against the queues."""
    scene = cb.Scene.from_desc(_chain())
    images, counts = [], []
    for queues in (False, True):
        r = cb.PBRenderer(cb.RenderingMethod.PATHTRACER)
        r.set_output_size(w, h)
        r.register_scene(scene)
        r.set_max_trace_depth(6)
        r.set_profiling(queues)
        r.render(cb.Camera.look_at((0, 0, 0), (1, 0.5, -1), (0, 1, 0), 70.0, w, h), 2)
        images.append(r.get_output_image())
        st = r.stats()
        counts.append((st["extension_rays"], st["shadow_rays"]))
    print(f"{w}x{h}: {counts}", flush=True)
    assert counts[0] == counts[1] and counts[0][1] > 0
    assert np.array_equal(images[0], images[1], equal_nan=True)
