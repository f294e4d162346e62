"""The workloads this renderer core is timed on: what its users have it do, through the Python
front end, from single-frame previews to the 1080p / 64-spp frame of the 1M-triangle scene.

listed() names twelve cases, draw() gives more of the same ranges; prepare() makes a case's inputs
and handles from a seed, run() is one pass, exact() the same outputs in 64 bits where they have a
64-bit value, and work() the bytes and operations a pass cannot do without. A Monte Carlo image
has no such value: its paths are defined by 32-bit random decisions.
"""
import ctypes
import math

import numpy as np
import torch

import cupbr_amd as cb
from cupbr_amd import scenes
from cupbr_amd.autograd import GridRender


def listed():
    return [
        # a picking or range-finding tool's batch: a few thousand closest-hit rays
        dict(name="queries_2k", kind="queries", scene="meshes", n=2048, visibility=False),
        # an external integrator's batches: incoherent closest hits, then their visibility tests
        dict(name="queries_1m", kind="queries", scene="boxes", n=1000003, visibility=True),
        # interactive preview: one frame of a small scene, read back by the host
        dict(name="path_cornell_256_1spp", kind="render", method="path", scene="cornell", width=256, height=256,
             spp=1, depth=5, roulette=False, readback=True, cache=False),
        # an odd-sized preview of every primitive and material with an environment, with roulette
        dict(name="path_mixed_331x217_6spp", kind="render", method="path", scene="mixed", width=331, height=217,
             spp=6, depth=8, roulette=True, readback=False, cache=False),
        # interactive camera moves in the large scene: one full-HD frame at a time
        dict(name="path_million_1080p_1spp", kind="render", method="path", scene="million", width=1920, height=1080,
             spp=1, depth=8, roulette=False, readback=False, cache=False),
        # the headline frame
        dict(name="path_million_1080p_64spp", kind="render", method="path", scene="million", width=1920, height=1080,
             spp=64, depth=8, roulette=False, readback=False, cache=False),
        # gradient-domain rendering with its reconstruction
        dict(name="gradient_cornell_512_16spp", kind="render", method="gradient", scene="cornell", width=512,
             height=512, spp=16, depth=5, roulette=False, readback=False, cache=False),
        # homogeneous media inside and outside objects
        dict(name="volume_512_16spp", kind="render", method="volume", scene="volumes", width=512, height=512, spp=16,
             depth=8, roulette=False, readback=False, cache=False),
        # one step of inverse rendering: forward render of a voxel medium and its gradients
        dict(name="grid_gradient_256_64spp", kind="grid", res=64, width=256, height=256, spp=64, depth=6,
             gradient=True),
        # radiance-cache predictions for about a frame's worth of path vertices
        dict(name="cache_infer_1m", kind="infer", n=1000003),
        # the cache's online training between frames
        dict(name="cache_train_16k_16", kind="train", rows=100003, batch=16384, steps=16),
        # post chain of a full-HD frame: 5-level bloom and tone map
        dict(name="post_1080p_gaussian", kind="post", width=1920, height=1080, pyramid=1, tone=0),
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of its range."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["queries", "render", "render", "render", "grid", "infer", "train", "post"])
    if kind == "queries":
        return dict(kind=kind, scene=rng.choice(["meshes", "boxes"]), n=_size(rng, 64, 2000000),
                    visibility=rng.random() < 0.5)
    if kind == "render":
        method = rng.choice(["path", "path", "path", "gradient", "volume", "ray"])
        w, h = _size(rng, 16, 1920), _size(rng, 16, 1080)
        most = 32e6 / (w * h * (5 if method == "gradient" else 1))
        spp = 1 if method == "ray" else _size(rng, 1, max(1, min(64, most)))
        if method == "gradient":
            scene = "cornell"
        elif method == "volume":
            scene = "volumes"
        else:
            scene = rng.choice(["cornell", "mixed", "boxes", "million"])
        cache = method == "path" and scene == "boxes" and rng.random() < 0.5
        return dict(kind=kind, method=method, scene=scene, width=w, height=h, spp=spp, depth=rng.randint(2, 9),
                    roulette=method in ("path", "volume") and rng.random() < 0.3, readback=rng.random() < 0.3,
                    cache=cache)
    if kind == "grid":
        return dict(kind=kind, res=_size(rng, 8, 96), width=_size(rng, 16, 256), height=_size(rng, 16, 256),
                    spp=_size(rng, 1, 64), depth=rng.randint(1, 8), gradient=rng.random() < 0.7)
    if kind == "infer":
        return dict(kind=kind, n=_size(rng, 1, 2000000))
    if kind == "train":
        return dict(kind=kind, rows=_size(rng, 100, 262144), batch=512 * _size(rng, 1, 64), steps=_size(rng, 1, 32))
    return dict(kind=kind, width=_size(rng, 16, 3840), height=_size(rng, 16, 2160), pyramid=rng.randint(0, 1),
                tone=rng.randint(0, 2))


# ------------------------------------------------------------------ inputs
_scenes = {}


def _scene(name):
    """(Scene on the GPU, camera arguments): a program loads a scene once and renders many views."""
    if name not in _scenes:
        if name == "meshes":
            desc, cam = scenes.random_mesh_scene(), None
        elif name == "boxes":
            desc, cam = scenes.million_triangles(n_spheres=5, subdiv=5, n_boxes=1000)
        elif name == "million":
            desc, cam = scenes.million_triangles()
        elif name == "cornell":
            desc, cam = scenes.cornell_box()
        elif name == "mixed":
            desc, cam = scenes.mixed_primitives()
        else:
            desc, cam = scenes.volume_spheres(), dict(eye=(0, 0, 0), target=(0, 0, 1), up=(0, 1, 0), vfov=90.0)
        s = cb.Scene.from_desc(desc)
        s.upload()
        _scenes[name] = (s, cam)
    return _scenes[name]


class _Buffer:
    """A device buffer of the library, for torch.as_tensor."""

    def __init__(self, ptr, shape, kind):
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=kind, data=(int(ptr), False), version=2)


def _tensor(owner, ptr, shape, kind="<f4"):
    """A buffer of `owner` (a renderer or a post-chain object) as a tensor, which keeps its owner: the
    buffer is freed with it."""
    t = torch.as_tensor(_Buffer(ptr, shape, kind), device="cuda")
    t.owner = owner
    return t


def _camera(cam, rng, w, h):
    """The scene's camera, moved a little by the seed (a few thousandths of its distance to the target)."""
    eye, target = np.asarray(cam["eye"], float), np.asarray(cam["target"], float)
    step = 0.005 * np.linalg.norm(target - eye)
    return cb.Camera.look_at(eye + rng.uniform(-step, step, 3), target + rng.uniform(-step, step, 3), cam["up"],
                             cam["vfov"], w, h)


def _rays(case, seed):
    """Incoherent rays from inside the scene's bounds: origins [n, 3], unit directions and distances."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = case["n"]
    lo, hi = (-10.0, 10.0) if case["scene"] == "meshes" else (0.0, 100.0)
    o = lo + (hi - lo) * torch.rand(n, 3, generator=g, device="cuda")
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1)
    dist = (0.05 + 0.5 * torch.rand(n, generator=g, device="cuda")) * (hi - lo)
    return torch.cat([o, d], 1).contiguous(), dist


def _cache_rows(n, seed, targets):
    """Records as path vertices leave them: position in the box, unit directions, roughness, albedos (and,
    for training, a radiance with a long tail)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    unit = lambda: torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1)  # noqa: E731
    r = lambda k: torch.rand(n, k, generator=g, device="cuda")  # noqa: E731
    cols = [100.0 * r(3), unit(), unit(), 0.05 + 0.95 * r(1), 0.1 + 0.8 * r(3), 0.9 * r(3)]
    if targets:
        cols += [torch.exp(0.7 * torch.randn(n, 3, generator=g, device="cuda") - 0.5), torch.zeros(n, 1, device="cuda")]
    return torch.cat(cols, 1).contiguous()


def _cache_weights(seed):
    """He-normal hidden layers and a small output layer."""
    rng = np.random.default_rng([seed, 5])
    return np.concatenate([rng.normal(0, math.sqrt(2 / 64), 4 * 4096), rng.normal(0, 0.1, 192)]).astype(np.float32)


def _cache(seed):
    c = cb.RadianceCache((0, 0, 0), (100, 100, 100))
    c.set_weights(_cache_weights(seed))
    return c


METHODS = dict(ray=cb.RenderingMethod.RAYTRACER, path=cb.RenderingMethod.PATHTRACER,
               gradient=cb.RenderingMethod.GRADIENTDOMAIN, volume=cb.RenderingMethod.VOLUME)


def _prepare_render(case, seed):
    w, h = case["width"], case["height"]
    scene, cam = _scene(case["scene"])
    r = cb.PBRenderer(METHODS[case["method"]])
    r.set_output_size(w, h)
    r.register_scene(scene)
    r.set_max_trace_depth(case["depth"])
    r.set_russian_roulette(case["roulette"])
    cache = None
    if case["cache"]:  # a trained cache, used without further training
        cache = _cache(seed)
        r.set_radiance_cache(cache, training_paths=0, train_steps=0)
    which = [cb.Image.OUTPUT]
    if case["method"] == "gradient":
        which += [cb.Image.BASE, cb.Image.GRADIENT_X, cb.Image.GRADIENT_Y]
    images = [_tensor(r, r.image_device_ptr(k), (h, w, 3)) for k in which]
    return dict(case=case, renderer=r, cache=cache, images=images,
                camera=_camera(cam, np.random.default_rng(seed), w, h))


def _prepare_grid(case, seed):
    g = scenes.grid_medium_scene(res=case["res"], width=case["width"], height=case["height"], seed=seed % 100003,
                                 target_seed=seed % 100003 + 1)
    cam = _camera(g["camera"], np.random.default_rng(seed), case["width"], case["height"])
    render = GridRender(cb.Scene.from_desc(g["desc"]), cam, cb.GridMedium.from_dict(g["density"].shape, g["medium"]),
                        case["width"], case["height"], spp=case["spp"], max_depth=case["depth"])
    # densities strictly inside (0, 1), as an optimiser keeps them
    density = torch.from_numpy(g["density"]).cuda().clamp(0.01, 0.99).requires_grad_(case["gradient"])
    albedo = torch.from_numpy(g["albedo"]).cuda().requires_grad_(case["gradient"])
    gen = torch.Generator(device="cuda").manual_seed(seed)
    weight = torch.randn(case["height"], case["width"], 3, generator=gen, device="cuda")
    return dict(case=case, render=render, density=density, albedo=albedo, weight=weight)


def _prepare_post(case, seed):
    w, h = case["width"], case["height"]
    post, tone = cb.PostProcessor(), cb.ToneMapper(cb.ToneMappingType(case["tone"]))
    hdr = _hdr(case, seed)
    torch.cuda.synchronize()
    post.set_bloom_pyramid(cb.BloomPyramid(case["pyramid"]))
    post.register_image(hdr.data_ptr(), w, h)
    tone.register_image(hdr.data_ptr(), w, h)
    p = ctypes.c_void_p()
    assert cb.lib().cupbr_tonemapper_get_render_buffer_device(tone._h, ctypes.byref(p)) == 0
    return dict(case=case, hdr=hdr, post=post, tone=tone, curve=cb.threshold_curve(1.0, 1.0),
                bloomed=_tensor(post, post.buffer_device_ptr(), (h, w, 3)),
                shown=_tensor(tone, p.value, (h, w, 4), "|u1"))


def _hdr(case, seed):
    """An HDR frame: log-normal radiance, a few pixels far above the bloom threshold."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.exp(torch.randn(case["height"], case["width"], 3, generator=g, device="cuda") - 0.7).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "queries":
        rays, dist = _rays(case, seed)
        return dict(case=case, scene=_scene(case["scene"])[0], rays=rays, dist=dist)
    if kind == "render":
        return _prepare_render(case, seed)
    if kind == "grid":
        return _prepare_grid(case, seed)
    if kind == "infer":
        return dict(case=case, cache=_cache(seed), inputs=_cache_rows(case["n"], seed, False))
    if kind == "train":
        return dict(case=case, cache=_cache(seed), rows=_cache_rows(case["rows"], seed, True))
    return _prepare_post(case, seed)


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "queries":
        out = list(s["scene"].trace_closest(s["rays"]))
        if case["visibility"]:
            out.append(s["scene"].trace_visibility(s["rays"], s["dist"]))
        return out
    if kind == "render":
        r = s["renderer"]
        r.reset()  # a new view: the running mean starts over
        r.render(s["camera"], case["spp"])
        if case["readback"]:
            return r.get_output_image()
        r.synchronize()  # the frame is used on the device next; render() runs on the renderer's own stream
        return s["images"]
    if kind == "grid":
        if not case["gradient"]:
            return s["render"](s["density"], s["albedo"])
        image = s["render"](s["density"], s["albedo"])
        return [image.detach(), *torch.autograd.grad(image, (s["density"], s["albedo"]), s["weight"])]
    if kind == "infer":
        return s["cache"].infer(s["inputs"])
    if kind == "train":
        loss = s["cache"].train(s["rows"], case["batch"], case["steps"], return_loss=True)
        return [loss, s["cache"].get_weights()]
    s["tone"].tone_map_bloom(s["post"], s["curve"])
    return [s["bloomed"], s["shown"]]


# ------------------------------------------------------------------ 64-bit values
def _exact_closest(case, seed):
    """Closest hits by testing every ray against every triangle and sphere of the mesh scene."""
    desc = scenes.random_mesh_scene()
    rays, _ = _rays(case, seed)
    o, d = rays[:, :3].double(), rays[:, 3:].double()
    tri = torch.from_numpy(desc["tris"]).cuda().double()
    v, e1, e2 = tri[:, :3], tri[:, 3:6] - tri[:, :3], tri[:, 6:] - tri[:, :3]
    ball = torch.from_numpy(desc["params"][desc["types"] == scenes.SPHERE]).cuda().double()
    best = torch.full((len(o),), math.inf, dtype=torch.float64, device="cuda")
    step = 2048
    for i in range(0, len(o), step):
        a, b = o[i:i + step, None], d[i:i + step, None]
        for k in range(0, len(v), 4096):
            f1, f2 = e1[None, k:k + 4096], e2[None, k:k + 4096]
            p = torch.linalg.cross(b.expand(-1, f2.shape[1], -1), f2.expand(len(b), -1, -1))
            det = (f1 * p).sum(-1)
            tv = a - v[None, k:k + 4096]
            u = (tv * p).sum(-1) / det
            q = torch.linalg.cross(tv, f1.expand(len(b), -1, -1))
            w = (b * q).sum(-1) / det
            t = (f2 * q).sum(-1) / det
            ok = (det.abs() >= 1e-5) & (u >= 0) & (u <= 1) & (w >= 0) & (u + w <= 1) & (t >= 0)
            t = torch.where(ok, t, torch.inf).amin(1)
            best[i:i + step] = torch.minimum(best[i:i + step], t)
        oc = a - ball[None, :, :3]
        h = (b * oc).sum(-1)
        disc = h * h - ((oc * oc).sum(-1) - ball[None, :, 3] ** 2)
        root = torch.sqrt(disc.clamp(min=0))
        t = torch.where(-h - root >= 0, -h - root, -h + root)
        t = torch.where((disc > 0) & (t >= 0), t, torch.inf).amin(1)
        best[i:i + step] = torch.minimum(best[i:i + step], t)
    return best


def _encode(x):
    """The cache's 64 input features, from records of 16 values; the box is [0, 100]^3."""
    pos = x[:, :3] / 100.0
    feats = []
    for a in range(3):
        for k in range(6):
            feats += [torch.sin(2.0 ** k * math.pi * pos[:, a]), torch.cos(2.0 ** k * math.pi * pos[:, a])]
    for c in (3, 6):
        for y in (torch.acos(x[:, c + 2].clamp(-1, 1)) / math.pi,
                  (torch.atan2(x[:, c + 1], x[:, c]) / math.pi + 1) / 2):
            for k in range(2):
                feats += [torch.sin(2.0 ** k * math.pi * y), torch.cos(2.0 ** k * math.pi * y)]
    feats += [1 - torch.exp(-x[:, 9])] + [x[:, 10 + k] for k in range(6)]
    one = torch.ones_like(x[:, 0])
    return torch.stack(feats + [one] + [torch.zeros_like(one)] * 4, 1)


def _layers(w):
    return [w[4096 * k:4096 * (k + 1)].reshape(64, 64) for k in range(4)] + [w[4 * 4096:].reshape(3, 64)]


def _mlp(w, x):
    for m in _layers(w)[:4]:
        x = torch.relu(x @ m.T)
    return x @ _layers(w)[4].T


def _hash32(x):
    m = 0xFFFFFFFF
    x = x & m
    x = x ^ (x >> 16)
    x = (x * 0x7FEB352D) & m
    x = x ^ (x >> 15)
    x = (x * 0x846CA68B) & m
    return x ^ (x >> 16)


def _exact_train(case, seed):
    """Adam (0.9, 0.99) on the relative L2 loss, over the batches the cache draws by hash."""
    rows = _cache_rows(case["rows"], seed, True).double()
    feats, target = _encode(rows[:, :16]), rows[:, 16:19]
    w = torch.from_numpy(_cache_weights(seed)).cuda().double()
    m, v, losses = torch.zeros_like(w), torch.zeros_like(w), []
    q = torch.arange(case["batch"], device="cuda")
    for step in range(1, case["steps"] + 1):
        pick = _hash32(q + (step * 0x9E3779B9 + 0x51ED270B)) % case["rows"]
        w.requires_grad_(True)
        y = _mlp(w, feats[pick])
        loss = ((y - target[pick]) ** 2 / (y.detach() ** 2 + 0.01)).sum()
        grad = torch.autograd.grad(loss, w)[0] / case["batch"]
        losses.append(loss.detach())
        m = 0.9 * m + 0.1 * grad
        v = 0.99 * v + 0.01 * grad * grad
        w = w.detach() - 1e-3 * (m / (1 - 0.9 ** step)) / (torch.sqrt(v / (1 - 0.99 ** step)) + 1e-10)
    return [torch.stack(losses), w]


def _at(img, x, y):
    """img[y, x] with both clamped to the image."""
    return img[y.clamp(0, img.shape[0] - 1)][:, x.clamp(0, img.shape[1] - 1)]


def _exact_bloom(case, seed):
    hdr = _hdr(case, seed).double()
    h, w = hdr.shape[:2]
    b = hdr.amax(2, keepdim=True)  # threshold 1, knee 1: curve (1, 0, 2, 0.25)
    soft = 0.25 * b.clamp(0, 2) ** 2
    low = hdr * torch.maximum(soft, b - 1) / b.clamp(min=1e-5)
    ar = lambda n: torch.arange(n, device="cuda")  # noqa: E731
    if case["pyramid"] == 0:
        x, y = ar(w // 2), ar(h // 2)
        half = sum(_at(low, 2 * x + i, 2 * y + j) for i in (0, 1) for j in (0, 1)) / 4
        tent = [1, 2, 1]
        up = sum(tent[i + 1] * tent[j + 1] * _at(half, ar(w) // 2 + i, ar(h) // 2 + j) for i in (-1, 0, 1)
                 for j in (-1, 0, 1))
        return hdr + up / 16 + low
    taps, level = [1, 4, 6, 4, 1], [low]
    for _ in range(5):
        s = level[-1]
        x, y = ar((s.shape[1] + 1) // 2), ar((s.shape[0] + 1) // 2)
        level.append(sum(taps[i] * taps[j] * _at(s, 2 * x + i - 2, 2 * y + j - 2) for i in range(5)
                         for j in range(5)) / 256)
    u = level[5]
    for k in (4, 3, 2, 1, 0):
        x, y = ar(level[k].shape[1]), ar(level[k].shape[0])
        u = level[k] + sum(_at(u, x // 2 + i * (x % 2), y // 2 + j * (y % 2)) for i in (0, 1) for j in (0, 1)) / 4
    return hdr + u / 6


def exact(case, seed):
    kind = case["kind"]
    if kind == "queries" and case["scene"] == "meshes" and case["n"] <= 65536:
        return [None, None, _exact_closest(case, seed)] + [None] * case["visibility"]
    if kind == "infer":
        w = torch.from_numpy(_cache_weights(seed)).cuda().double()
        return _mlp(w, _encode(_cache_rows(case["n"], seed, False).double()))
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "post":
        return [_exact_bloom(case, seed), None]
    return None


# ------------------------------------------------------------------ work
# Rays per camera path, and bytes of BVH nodes and primitives, of each scene; a ray costs about 100
# operations per node (four slab tests) and 60 per primitive it has to look at.
SCENE = dict(meshes=(1, 12, 10, 0.9e6), boxes=(5, 18, 7, 9e6), million=(6.5, 25, 8, 75e6), cornell=(9, 4, 6, 3e3),
             mixed=(7, 2, 8, 3e3), volumes=(9, 1, 8, 2e3))


def work(case):
    kind = case["kind"]
    if kind == "queries":
        _, nodes, prims, size = SCENE[case["scene"]]
        rays = case["n"] * (2 if case["visibility"] else 1)
        return dict(bytes=case["n"] * (36 + (29 if case["visibility"] else 0)) + min(size, rays * nodes * 128),
                    flops=rays * (100 * nodes + 60 * prims))
    if kind == "render":
        per, nodes, prims, size = SCENE[case["scene"]]
        px = case["width"] * case["height"]
        paths = px * case["spp"] * (5 if case["method"] == "gradient" else 1)
        images = 8 if case["method"] == "gradient" else 1
        per = 2 if case["method"] == "ray" else min(per, 2 * case["depth"])
        return dict(bytes=12 * px * images + size, flops=paths * per * (100 * nodes + 60 * prims + 200))
    if kind == "grid":
        px, voxels = case["width"] * case["height"], case["res"] ** 3
        events = px * case["spp"] * (25 if case["gradient"] else 10)  # grid points looked up
        return dict(bytes=(24 if case["gradient"] else 12) * px + voxels * (8 if case["gradient"] else 4),
                    flops=events * (100 if case["gradient"] else 50))
    if kind == "infer":
        return dict(bytes=case["n"] * (64 + 12) + 4 * cb.NRC_PARAMS, flops=case["n"] * 2.0 * cb.NRC_PARAMS)
    if kind == "train":
        rows = min(case["rows"], case["batch"] * case["steps"])
        return dict(bytes=rows * 80 + 12 * cb.NRC_PARAMS, flops=case["batch"] * case["steps"] * 6.0 * cb.NRC_PARAMS)
    px = case["width"] * case["height"]
    return dict(bytes=px * (12 + 12 + 4), flops=px * 120)
