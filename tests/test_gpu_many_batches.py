"""More batches than a launch has workgroups to give one to each (2^24 of 256
threads): the cloud is made and drawn as before it had group bounds."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc


@pytest.mark.gpu
def test_two_to_the_24_batches(ctx):
    xyz, rgba = orc.generate(pcr.gen_cfg(pcr.SCENE_CITY, 20_000, seed=8, num_buildings=9))
    perm = orc.morton_order(xyz)[0]
    b, lo, med, hi = pcr.encode_batches_host(xyz[perm], 500)
    nb = (1 << 24) + 3
    many = np.zeros(nb, b.dtype)
    many["parent"] = -1
    for k in ("min", "max"):
        many[k] = -1.0e7   # empty batches, outside every view
    at = np.linspace(0, nb - 1, len(b)).astype(np.int64)   # the first and the last among them
    many[at] = b
    v = pcr.look_at((150, -420, 260), (150, 150, 10), up=(0, 0, 1), near=1, far=3000, width=333, height=211)
    ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
    assert (ref != np.uint64(0xFFFFFFFFFFFFFFFF)).sum() > 1000
    cloud = ctx.upload_batched(many, lo, med, hi, rgba[perm])
    del many
    fb = ctx.framebuffer(v.width, v.height)
    for _ in range(2):
        ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2), fb)
        assert np.array_equal(fb.keys(), ref)
    fb.close()
    cloud.close()
