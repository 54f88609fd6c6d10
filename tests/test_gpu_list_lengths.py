"""Lists of drawn batches around the number of workgroups of a launch (about
1,000 to 2,000), where the batches are shared out in two, three or four parts,
sorted and unsorted: frames equal the oracle's (hqs: the direct passes')."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc
from test_gpu_groups import layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batches", [520, 700, 980, 1300, 1450, 1700, 2200, 4100])
@pytest.mark.parametrize("shuffle", [False, True])
def test_every_point_is_drawn_once(ctx, batches, shuffle):
    size = 1500   # two rounds of a workgroup: parts three and four are empty
    n = batches * size - 700
    b, lo, med, hi, rgba = layout(n, size, False, shuffle)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    v = pcr.look_at((150, -420, 260), (150, 150, 10), up=(0, 0, 1), near=1, far=3000, width=477, height=301)
    ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
    direct = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
    ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=0), direct)
    href = direct.hqs()
    for block, tile_px in ((256, 2048), (128, 1024)):
        fb = ctx.framebuffer(v.width, v.height)
        ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, block_size=block, tile_px=tile_px), fb)
        assert np.array_equal(fb.keys(), ref)
        fb.close()
        # hqs sums count a point that is drawn twice
        hq = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, block_size=block, tile_px=tile_px), hq)
        assert all(np.array_equal(a, r) for a, r in zip(hq.hqs(), href))
        hq.close()
        fbs = [ctx.framebuffer(v.width, v.height, pcr.FB_HQS) for _ in range(3)]
        mv = pcr.MultiView(ctx, cloud, [v] * 3, fbs, pcr.params(pcr.MODE_HQS), tune=pcr.Tune(block, 40, 0, tile_px))
        mv.launch()
        for f in fbs:
            assert all(np.array_equal(a, r) for a, r in zip(f.hqs(), href))
        mv.close()
        for f in fbs:
            f.close()
    direct.close()
    cloud.close()
