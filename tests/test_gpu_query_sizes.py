"""Batch queries of every size give the same results.

Batches are traced by 64, 32 or 16 lanes per ray, or one, according to their size. Each ray's closest
hit and visibility is the same whatever else is in the batch, so any slice of a large batch must equal
the slice of the large batch's results, bit for bit; small batches are also compared with the oracle.
"""
import numpy as np
import pytest

import cupbr_amd as cb
import oracle
from cupbr_amd import scenes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SCENES = {
    "meshes": (lambda: scenes.random_mesh_scene(), -12.0, 12.0),
    "soup": (lambda: scenes.random_triangle_soup(3000, seed=5), -12.0, 12.0),
    "cornell": (lambda: scenes.cornell_box()[0], 0.0, 1.0),
    "boxes": (lambda: scenes.cornell_box(as_triangles=False)[0], 0.0, 1.0),
    "mixed": (lambda: scenes.mixed_primitives()[0], -3.0, 3.0),
}


def _rays(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(lo, hi, (n, 3))
    d = rng.normal(size=(n, 3))
    d[::17, 0] = 0.0  # rays in coordinate planes and along axes
    d[::34, 1] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, d], 1).astype(np.float32), rng.uniform(0.0, hi - lo, n).astype(np.float32)


@pytest.mark.parametrize("name", list(SCENES))
def test_batch_sizes_agree(name):
    make, lo, hi = SCENES[name]
    desc = make()
    S = cb.Scene.from_desc(desc)
    n = 163_841
    rays, dist = _rays(n, lo, hi, 11)
    rays_d, dist_d = torch.from_numpy(rays).cuda(), torch.from_numpy(dist).cuda()
    obj, tri, t = (x.cpu().numpy() for x in S.trace_closest(rays_d))
    vis = S.trace_visibility(rays_d, dist_d).cpu().numpy()
    assert (obj >= 0).any() and (vis == 0).any() and (vis != 0).any()
    for first, count in ((0, 1), (5, 3), (0, 64), (1000, 8191), (1, 8192), (7, 8193), (300, 32768), (4000, 32769),
                         (0, 163_840)):
        part = slice(first, first + count)
        print(f"{name}: {count} rays", flush=True)
        o2, r2, t2 = (x.cpu().numpy() for x in S.trace_closest(rays_d[part].contiguous()))
        v2 = S.trace_visibility(rays_d[part].contiguous(), dist_d[part].contiguous()).cpu().numpy()
        assert np.array_equal(obj[part], o2) and np.array_equal(tri[part], r2) and np.array_equal(vis[part], v2)
        assert np.array_equal(t[part].view(np.uint32), t2.view(np.uint32))
    ref = oracle.OracleScene(desc, precisions=(32,))
    ro, rt, rd = ref.trace(rays[:4096], precision=32, mode=0)
    assert np.array_equal(ro, obj[:4096]) and np.array_equal(rt, tri[:4096]) and np.array_equal(rd, t[:4096])
    assert np.array_equal(ref.visibility(rays[:4096], dist[:4096], precision=32, mode=0), vis[:4096])


def test_scene_without_a_tree():
    """Only planes and quads, which are tested outside the tree."""
    b = scenes.SceneBuilder()
    for k in range(70):  # more of them than a wave has lanes
        b.quad((0.01 * k, 0.3, 0.5), (0, 0, 1), (0.02, 0, 0), (0, 0.05, 0), scenes.material())
    b.plane((0, -1, 0), (0, 1, 0), scenes.material())
    b.point_light((0, 5, 0), (10, 10, 10))
    desc = b.desc()
    S = cb.Scene.from_desc(desc)
    ref = oracle.OracleScene(desc, precisions=(32,))
    rays, dist = _rays(100, 0.0, 1.0, 3)
    for n in (1, 100):
        got = [x.cpu().numpy() for x in S.trace_closest(torch.from_numpy(rays[:n]).cuda())]
        for a, c in zip(ref.trace(rays[:n], precision=32, mode=0), got):
            assert np.array_equal(a, c)
        vis = S.trace_visibility(torch.from_numpy(rays[:n]).cuda(), torch.from_numpy(dist[:n]).cuda()).cpu().numpy()
        assert np.array_equal(ref.visibility(rays[:n], dist[:n], precision=32, mode=0), vis)


@pytest.mark.parametrize("name", ["meshes", "mixed"])
def test_large_batches_agree(name):
    """One lane per ray: pieces of 64 rays (one refill) to 512, whole and ragged, with the wave's last rays
    walked by groups; the results of a batch are the slice of a larger one's."""
    make, lo, hi = SCENES[name]
    S = cb.Scene.from_desc(make())
    n = 2_200_001
    rays, dist = (torch.from_numpy(x).cuda() for x in _rays(n, lo, hi, 23))
    whole = list(S.trace_closest(rays)) + [S.trace_visibility(rays, dist)]
    for first, count in ((0, 64), (3, 100_000), (n - 163_841, 163_841), (1, 262_144), (17, 700_003)):
        print(f"{name}: {count} rays", flush=True)
        part = slice(first, first + count)
        r, d = rays[part].contiguous(), dist[part].contiguous()
        for a, b in zip(whole, list(S.trace_closest(r)) + [S.trace_visibility(r, d)]):
            assert torch.equal(a[part].view(torch.uint8), b.view(torch.uint8))
