"""Multi-view launches of clouds with group bounds: pairs of near-identical
views (drawn together), views of other sizes (drawn one at a time), short lists
split into many parts, odd batch sizes and unaligned starts. Every view's
framebuffer equals the oracle's (hqs: the direct passes' of that view)."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from test_gpu_groups import layout, views

pytestmark = pytest.mark.gpu

LAYOUTS = [(70, 1, True, False), (1000, 63, True, False), (1000, 64, False, False), (9001, 1023, True, False),
           (9001, 1024, False, False), (20011, 1025, True, False), (150_001, 10240, True, False),
           (150_001, 16385, True, True), (200_003, 200_003, True, False)]


def eyes():
    """Pairs 0.05 apart of the first two views of the single-view tests, then
    all of those views."""
    out = []
    up = (0, 0, 1)
    for s in (0.0, 0.05):
        out.append(pcr.look_at((150 + s, -420, 260), (150 + s, 150, 10), up=up, near=1, far=3000, width=333, height=211))
    for s in (0.0, 0.05):
        out.append(pcr.look_at((150 + s, -9000, 6000), (150 + s, 150, 0), up=up, near=1, far=30000, width=640, height=480))
    return out + list(views())


@pytest.mark.parametrize("n,size,shift,shuffle", LAYOUTS)
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128)])
def test_multiview_raster_equals_oracle(ctx, n, size, shift, shuffle, tile_px, block):
    from oracle import orc
    b, lo, med, hi, rgba = layout(n, size, shift, shuffle)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    vs = eyes()
    refs = [orc.render_batched(b, lo, med, hi, v, 1)[0] for v in vs]
    for skip in (True, False):
        fbs = [ctx.framebuffer(v.width, v.height) for v in vs]
        prm = pcr.params(pcr.MODE_LAS2, occlusion_skip=skip)
        mv = pcr.MultiView(ctx, cloud, vs, fbs, prm, tune=pcr.Tune(block, 40, 0, tile_px))
        for _ in range(3):
            mv.launch()
            for fb, ref in zip(fbs, refs):
                assert np.array_equal(fb.keys(), ref), f"{fb.width}x{fb.height}: {(fb.keys() != ref).sum()} keys differ"
        mv.close()
        for fb in fbs:
            fb.close()
    cloud.close()


@pytest.mark.parametrize("n,size,shift,shuffle", LAYOUTS[1:])
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128)])
def test_multiview_hqs_equals_the_direct_passes(ctx, n, size, shift, shuffle, tile_px, block):
    b, lo, med, hi, rgba = layout(n, size, shift, shuffle)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    vs = eyes()
    refs = []
    for v in vs:
        fb = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=0), fb)
        refs.append(fb.hqs())
        fb.close()
    for skip in (True, False):
        fbs = [ctx.framebuffer(v.width, v.height, pcr.FB_HQS) for v in vs]
        prm = pcr.params(pcr.MODE_HQS, occlusion_skip=skip)
        mv = pcr.MultiView(ctx, cloud, vs, fbs, prm, tune=pcr.Tune(block, 40, 0, tile_px))
        for _ in range(2):
            mv.launch()
            for fb, ref in zip(fbs, refs):
                assert all(np.array_equal(a, r) for a, r in zip(fb.hqs(), ref))
        mv.close()
        for fb in fbs:
            fb.close()
    cloud.close()
