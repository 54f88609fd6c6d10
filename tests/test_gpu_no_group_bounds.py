"""The paths that are left when a cloud has no group bounds (the memory for them
was not there), and the point-by-point kernel of mode LAS at every workgroup
size: over odd batch sizes and unaligned starts, against the oracle."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc
from test_gpu_groups import layout, views

pytestmark = pytest.mark.gpu

LAYOUTS = [(70, 1, True, False), (1000, 63, True, False), (9001, 1024, False, False), (20011, 1025, True, False),
           (150_001, 10240, True, False), (150_001, 16385, True, True), (200_003, 200_003, True, False)]


def all_views():
    """Those of the grouped tests, and one from among the points (batches that
    reach behind the eye, rectangles many tiles high)."""
    return list(views()) + [pcr.look_at((150, 150, 12), (150, 260, 0), up=(0, 0, 1), near=0.01, far=3000, width=400, height=700)]


def upload(ctx, lay, bounds):
    cloud = ctx.upload_batched(*lay)
    if not bounds:
        lib = pcr.capi.load()
        assert lib.pcr_test_drop_group_bounds(cloud.h) == 0
    return cloud


@pytest.mark.parametrize("n,size,shift,shuffle", LAYOUTS)
def test_las_at_every_workgroup_size(ctx, n, size, shift, shuffle):
    lay = layout(n, size, shift, shuffle)
    for bounds in (True, False):
        cloud = upload(ctx, lay, bounds)
        for v in all_views():
            ref, _ = orc.render_batched(*lay[:4], v, 1)
            fb = ctx.framebuffer(v.width, v.height)
            for block in (0, 64, 128, 256, 512):
                ctx.render(cloud, v, pcr.params(pcr.MODE_LAS, block_size=block), fb)
                assert np.array_equal(fb.keys(), ref), (bounds, block)
            fb.close()
        cloud.close()


@pytest.mark.parametrize("n,size,shift,shuffle", LAYOUTS)
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
def test_frames_without_bounds(ctx, n, size, shift, shuffle, tile_px, block):
    lay = layout(n, size, shift, shuffle)
    cloud = upload(ctx, lay, False)
    vs = all_views()
    refs = [orc.render_batched(*lay[:4], v, 1)[0] for v in vs]
    hrefs = [orc.hqs_batched(*lay, v, 1) for v in vs]
    for v, ref, href in zip(vs, refs, hrefs):
        for skip in (True, False):
            prm = dict(tile_px=tile_px, block_size=block, occlusion_skip=skip)
            fb = ctx.framebuffer(v.width, v.height)
            for clear in (True, False):
                ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, clear_before=clear, **prm), fb)
                assert np.array_equal(fb.keys(), ref)
            fb.close()
            fb = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
            ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, **prm), fb)
            assert all(np.array_equal(a, r) for a, r in zip(fb.hqs(), href))
            fb.close()
    for mode, kind in ((pcr.MODE_LAS2, pcr.FB_KEY64), (pcr.MODE_HQS, pcr.FB_HQS)):
        fbs = [ctx.framebuffer(v.width, v.height, kind) for v in vs + vs[:1]]   # the last a pair of the first
        mv = pcr.MultiView(ctx, cloud, vs + vs[:1], fbs, pcr.params(mode), tune=pcr.Tune(block, 40, 0, tile_px))
        mv.launch()
        for k, fb in enumerate(fbs):
            if kind == pcr.FB_KEY64:
                assert np.array_equal(fb.keys(), refs[k % len(vs)])
            else:
                assert all(np.array_equal(a, r) for a, r in zip(fb.hqs(), hrefs[k % len(vs)]))
        mv.close()
        for fb in fbs:
            fb.close()
    cloud.close()
