"""Views from far outside the cloud, where the tiled raster draws batches whole
(a batch larger than the tile point by point), and the same cloud from nearby,
where it draws them in parts. Either way the keys are the oracle's."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc


def cloud_with_a_scattered_batch():
    """Small batches in Morton order, and every 20th over the whole scene."""
    xyz, rgba = orc.generate(pcr.gen_cfg(pcr.SCENE_CITY, 66_003, seed=3, num_buildings=9))
    perm = orc.morton_order(xyz)[0]
    size = 1024
    n = len(perm) // size
    scattered = np.arange(0, n, 20)
    pool = np.concatenate([np.arange(k * size, (k + 1) * size) for k in scattered])
    perm[pool] = perm[np.random.default_rng(4).permutation(pool)]
    b, lo, med, hi = pcr.encode_batches_host(xyz[perm], size)
    return b, lo, med, hi, rgba[perm]


@pytest.mark.gpu
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
@pytest.mark.parametrize("dist", [0.6, 2.0, 8.0, 30.0])
def test_far_views_equal_oracle(ctx, tile_px, block, dist):
    b, lo, med, hi, rgba = cloud_with_a_scattered_batch()
    mid = 0.5 * (b["min"].min(0) + b["max"].max(0))
    ext = float((b["max"].max(0) - b["min"].min(0)).max())
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    for az in (0.4, 2.5):
        eye = mid + dist * ext * np.array([np.cos(az), np.sin(az), 0.7])
        v = pcr.look_at(tuple(map(float, eye)), tuple(map(float, mid)), up=(0, 0, 1), near=1, far=1e6, width=643,
                        height=397)
        ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
        for skip in (True, False):
            fb = ctx.framebuffer(v.width, v.height)
            prm = dict(tile_px=tile_px, block_size=block, occlusion_skip=skip)
            ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, **prm), fb)
            assert np.array_equal(fb.keys(), ref)
            ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, clear_before=False, **prm), fb)
            assert np.array_equal(fb.keys(), ref) and ctx.stats().atomics_issued == 0
            fb.close()
        fb = ctx.framebuffer(v.width, v.height)
        ctx.render(cloud, v, pcr.params(pcr.MODE_LAS), fb)
        assert np.array_equal(fb.keys(), ref)
        fb.close()
    cloud.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,size", [(3000, 7), (70_003, 1024), (200_003, 10240)])
def test_unsorted_points_equal_oracle(ctx, n, size):
    """Points in a random order: every batch covers the scene, near and far."""
    xyz, rgba = orc.generate(pcr.gen_cfg(pcr.SCENE_TERRAIN, n, seed=5))
    perm = np.random.default_rng(6).permutation(n)
    b, lo, med, hi = pcr.encode_batches_host(xyz[perm], (size + 3) // 4 * 4)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba[perm])
    mid = 0.5 * (b["min"].min(0) + b["max"].max(0))
    ext = float((b["max"].max(0) - b["min"].min(0)).max())
    for dist in (0.0, 0.8, 20.0):   # inside, nearby, far
        eye = mid + np.array([0.3, -0.2, 0.1]) * ext * (0.3 + 2 * dist)
        v = pcr.look_at(tuple(map(float, eye)), tuple(map(float, mid)), up=(0, 0, 1), near=0.1, far=1e6, width=643, height=397)
        ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
        direct = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=0), direct)
        for mode in (pcr.MODE_LAS2, pcr.MODE_LAS):
            fb = ctx.framebuffer(v.width, v.height)
            for clear in (True, False):
                ctx.render(cloud, v, pcr.params(mode, clear_before=clear), fb)
                assert np.array_equal(fb.keys(), ref)
            fb.close()
        hq = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(pcr.MODE_HQS), hq)
        assert all(np.array_equal(a, r) for a, r in zip(hq.hqs(), direct.hqs()))
        hq.close()
        direct.close()
    cloud.close()
