"""What the tiled kernels leave out and how pcr_stats counts it: groups behind a
wall, batches behind it as a whole, parts outside the image."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc

pytestmark = pytest.mark.gpu
N = 10240   # points of the wall and of the block behind it, a batch each
CLEAR = np.uint64(0xFFFFFFFFFFFFFFFF)


def scene(wall_to):
    """A wall at z = 2 over x in [-1.5, wall_to], and a block of points behind
    it over x in [-1.5, 1.5], in Morton order."""
    u, v = np.meshgrid(np.linspace(-1.5, wall_to, 80), np.linspace(-1.5, 1.5, 128), indexing="ij")
    wall = np.stack([u, v, np.full(u.shape, 2.0)], -1).reshape(-1, 3).astype(np.float32)
    block = np.random.default_rng(7).uniform((-1.5, -1.5, -3), (1.5, 1.5, -1), (N, 3)).astype(np.float32)
    block = block[orc.morton_order(block)[0]]
    b, lo, med, hi = pcr.encode_batches_host(np.concatenate([wall, block]), N)
    assert len(b) == 2 and b["num_points"].tolist() == [N, N]
    return b, lo, med, hi, np.arange(2 * N, dtype=np.uint32)


def front():
    return pcr.look_at((0, 0, 10), (0, 0, 0), up=(0, 1, 0), fovy=60.0, near=0.1, far=100, width=128, height=128)


@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
def test_groups_behind_half_a_wall(ctx, tile_px, block):
    """Half of the block's points lie behind the wall: with the wall drawn, the
    groups that do not touch the edge or the front are left out, at least a
    fifth of the block (the leftmost two sixths of it, less its outermost
    groups), and no batch is skipped as a whole."""
    lay = scene(0.0)
    b, lo, med, hi, rgba = lay
    cloud, v = ctx.upload_batched(*lay), front()
    ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
    fb = ctx.framebuffer(v.width, v.height)
    ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block), fb)
    assert np.array_equal(fb.keys(), ref)
    ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block, clear_before=False), fb)
    st = ctx.stats()
    assert np.array_equal(fb.keys(), ref)
    assert N // 5 <= st.points_occluded < N and st.batches_occluded == 0
    assert st.bytes_occluded == 4 * st.points_occluded   # nothing lies outside the image
    fb.close()
    ref2 = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
    ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=0), ref2)
    hq = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
    ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=tile_px, block_size=block), hq)   # pass 2 knows the final depths
    st = ctx.stats()
    assert all(np.array_equal(a, r) for a, r in zip(hq.hqs(), ref2.hqs()))
    assert N // 5 <= st.points_occluded < 2 * N and st.batches_occluded == 0
    hq.close()
    ref2.close()
    cloud.close()


@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
def test_a_batch_behind_a_whole_wall_counts_once(ctx, tile_px, block):
    lay = scene(1.5)
    cloud, v = ctx.upload_batched(*lay), front()
    fb = ctx.framebuffer(v.width, v.height)
    ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block), fb)
    ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block, clear_before=False), fb)
    st = ctx.stats()
    # the block's rectangle: 1.5 * 64 / tan(30 deg) / 11 = 15.1 pixels to either side of the centre, a margin of one;
    # a batch over more pixels than the tile is skipped in runs of its parts, and is no skipped batch
    whole = 1 if 34 * 34 <= tile_px else 0
    assert (st.batches_occluded, st.points_occluded, st.bytes_occluded) == (whole, N, 4 * N)
    ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block, occlusion_skip=False), fb)
    st = ctx.stats()
    assert (st.batches_occluded, st.points_occluded, st.bytes_occluded) == (0, 0, 0)
    fb.close()
    cloud.close()


@pytest.mark.parametrize("mode", [pcr.MODE_LAS2, pcr.MODE_HQS, pcr.MODE_LAS])
def test_parts_outside_the_image_are_not_read(ctx, mode):
    """The block seen from nearby and from its right: a point is off the image
    where 4.5 - x > 0.77 depth (200 pixels of 260 per unit), at the farthest
    depth of 5 for x < 0.65. So the left half is. The bounds of a group that
    spans two cells of the Morton order are wide, so not all five parts of it
    are known to be, but the first is (within one cell, well off the image)."""
    b, lo, med, hi, rgba = scene(0.0)
    b, lo, med, hi, rgba = b[1:].copy(), lo[N:].copy(), med[N:].copy(), hi[N:].copy(), rgba[N:].copy()
    b["first_point"] = 0
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    v = pcr.look_at((4.5, 0, 2), (4.5, 0, 0), up=(0, 1, 0), fovy=60.0, near=0.1, far=100, width=400, height=300)
    hqs = mode == pcr.MODE_HQS
    fb = ctx.framebuffer(v.width, v.height, pcr.FB_HQS if hqs else pcr.FB_KEY64)
    ctx.render(cloud, v, pcr.params(mode, occlusion_skip=False), fb)
    st = ctx.stats()
    if hqs:
        ref = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(mode, tile_px=0), ref)
        assert all(np.array_equal(a, r) for a, r in zip(fb.hqs(), ref.hqs()))
        ref.close()
    else:
        assert np.array_equal(fb.keys(), orc.render_batched(b, lo, med, hi, v, 1)[0])
    per_point = 12 if hqs else 4   # hqs: the plane in both passes, the colour in the second
    assert st.points_occluded == 0 and st.batches_occluded == 0
    assert per_point * 1024 <= st.bytes_occluded < per_point * N and st.bytes_occluded % per_point == 0
    fb.close()
    cloud.close()
