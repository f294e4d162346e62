"""Gaussian-pyramid bloom and tone map at the edges of their tiles.

A frame is four launches of tiles (32 x 8 of level 1, 8 x 8 of level 3, 4 x 4 of level 5, 64 x 16 pixels); sizes on
both sides of each tile's edge, odd levels and images smaller than one tile, against the oracle: the image bit for
bit, bytes within one step (the host's powf) and equal to the unfused tone map's.
"""
import numpy as np
import pytest

import cupbr_amd as cb
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("w,h", [(2, 3), (3, 2), (5, 100), (63, 15), (64, 16), (65, 17), (127, 33), (129, 47), (255, 31),
                                 (257, 129), (31, 513), (640, 16)])
@pytest.mark.parametrize("kind", list(cb.ToneMappingType))
def test_gaussian_bloom_tile_edges(w, h, kind):
    rng = np.random.default_rng(w * 1000 + h)
    hdr = (rng.exponential(0.7, (h, w, 3)) * rng.choice([0.0, 0.2, 1.0, 30.0], (h, w, 1))).astype(np.float32)
    t = torch.from_numpy(hdr).cuda()
    curve = cb.threshold_curve(1.0, 0.5)
    post = cb.PostProcessor()
    post.set_bloom_pyramid(cb.BloomPyramid.GAUSSIAN5)
    post.register_image(t.data_ptr(), w, h)
    fused = cb.ToneMapper(kind)
    fused.register_image(t.data_ptr(), w, h)
    fused.tone_map_bloom(post, curve)
    want = oracle.bloom_gaussian(hdr, curve)
    assert np.array_equal(post.get_post_process_buffer(), want)
    tone = cb.ToneMapper(kind)
    tone.register_image(post.buffer_device_ptr(), w, h)
    tone.tone_map()
    got = fused.get_render_buffer()
    assert np.array_equal(got, tone.get_render_buffer())
    ref = oracle.tonemap(want, int(kind), 1.0).astype(np.int32)
    assert np.abs(got.astype(np.int32) - ref).max() <= 1


def test_tone_map_of_special_values():
    """Black, negative, saturated, infinite and NaN channels, and values at the steps of the bytes."""
    x = np.array([0.0, -0.0, -1.0, 1e-42, 1e-30, 0.0031308, 1.0, 20.0, 1e30, np.inf, -np.inf, np.nan], np.float32)
    steps = (np.arange(1, 256) / 255.0) ** 2.2
    x = np.concatenate([x, steps.astype(np.float32), -np.log1p(-np.minimum(steps, 1 - 1e-7)).astype(np.float32)])
    img = np.repeat(x[None, :, None], 3, axis=2)
    t = torch.from_numpy(img).cuda()
    for kind in cb.ToneMappingType:
        tm = cb.ToneMapper(kind)
        tm.register_image(t.data_ptr(), img.shape[1], 1)
        tm.tone_map()
        got, ref = tm.get_render_buffer().astype(np.int32), oracle.tonemap(img, int(kind), 1.0).astype(np.int32)
        finite = np.isfinite(x)
        assert np.abs(got - ref)[:, finite].max() <= 1, kind
        assert got[0, 0, 0] == 0 and (got[..., 3] == 255).all()


def test_bytes_of_every_float():
    """The fast route's byte is powf's for each of the 2^32 floats, infinities and NaN among them."""
    assert cb.tone_byte_check() == [0, 0, 0, 0]
