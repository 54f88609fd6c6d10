"""The tiled raster's group bounds: 64-point groups left out when the depths
under them are nearer, batches over more pixels than the tile drawn in parts,
short lists split into more parts, and the near-first slices of the list.

A group that is wrongly left out, a part that is cut at the wrong word or a
batch that is listed twice changes keys, so every framebuffer must equal the
oracle's bit for bit. The CPU half checks the bound itself: over random boxes
and views every point's pixel lies in its group's rectangle and no point is
nearer than the group's depth."""
import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc

F = np.float32


def fma(a, b, c):
    """float32 fma: the product is exact in float64, the sum rounds twice at most."""
    return (np.float64(a) * np.float64(b) + np.float64(c)).astype(F)


def project(t, p):
    rows = [fma(t[8 + k], p[2], fma(t[4 + k], p[1], fma(t[k], p[0], t[12 + k]))) for k in (0, 1, 3)]
    return rows


def group_rect(t, lo, hi, w, h, slack_px, slack_w):
    c, e = [F(0.5) * (lo[a] + hi[a]) for a in range(3)], [F(0.5) * np.abs(hi[a] - lo[a]) for a in range(3)]
    px, py, pw = project(t, c)
    ew = fma(e[2], abs(t[11]), fma(e[1], abs(t[7]), e[0] * abs(t[3])))
    iv, lw = F(1) / pw, pw - ew
    il, nx, ny = F(1) / lw, px * iv, py * iv
    r = [fma(e[2], np.abs(fma(-n, t[11], t[8 + k])), fma(e[1], np.abs(fma(-n, t[7], t[4 + k])),
             e[0] * np.abs(fma(-n, t[3], t[k])))) for k, n in ((0, nx), (1, ny))]
    fw, fh = F(0.5) * F(w), F(0.5) * F(h)
    m = np.maximum(np.maximum(np.abs(nx) + r[0] * il, np.abs(ny) + r[1] * il), F(1))
    s = slack_px * m
    cx, cy, dx, dy = fma(nx, fw, fw), fma(ny, fh, fh), fma(r[0] * il, fw, s), fma(r[1] * il, fh, s)
    wild = ~((m <= 64) & (ew <= F(0.5) * pw))
    return np.floor(cx - dx), np.floor(cy - dy), np.floor(cx + dx), np.floor(cy + dy), lw - slack_w, wild


@pytest.mark.parametrize("offset,extent", [(0.0, 100.0), (5000.0, 40.0), (-2000.0, 30.0), (1.0e5, 500.0)])
def test_group_bound_holds_its_points(offset, extent):
    rng = np.random.default_rng(int(extent))
    bounded = 0
    for _ in range(60):
        mn = (offset + rng.uniform(-extent, extent, 3)).astype(F)
        mx = (mn + rng.uniform(0.01, extent, 3).astype(F)).astype(F)
        mid = 0.5 * (mn + mx)
        eye = mid + rng.normal(size=3) * extent * rng.uniform(0.8, 6)
        W, H = int(rng.integers(3, 4000)), int(rng.integers(3, 3000))
        v = pcr.look_at(tuple(map(float, eye)), tuple(map(float, mid + rng.normal(size=3) * extent * 0.3)),
                        up=(0, 0, 1), near=0.01, far=1e6, width=W, height=H)
        t = np.array(v.transform[:], F)
        corners = np.array([[(mx if c >> a & 1 else mn)[a] for a in range(3)] for c in range(8)], F).T
        pwc = project(t, corners)[2]
        big = np.maximum(np.abs(mn), np.abs(mx))
        ex, ey, ew = (F(abs(t[12 + k]) + sum(abs(t[4 * a + k]) * big[a] for a in range(3))) for k in (0, 1, 3))
        side = F(max(W, H))
        spread = side * F(2.0 ** -21) * (max(ex, ey) + ew)
        wlo = F(pwc.min() - F(2.0 ** -18) * ew)
        if not (pwc.min() >= F(2.0 ** -12) + F(2.0 ** -16) * ew and pwc.min() >= spread and wlo > 0):
            continue
        bounded += 1
        slack_px, slack_w = spread / wlo + side * F(2.0 ** -19), F(2.0 ** -19) * ew
        q0 = rng.integers(0, 1024, (3, 400))
        q1 = np.minimum(q0 + rng.integers(0, 60, (3, 400)), 1023)
        q = np.array([rng.integers(q0, q1 + 1) for _ in range(64)])             # points x axes x groups
        scale = ((mx - mn) / F(1024)).astype(F)[:, None]
        dec = lambda k: fma(k.astype(F), scale, mn[:, None])
        x0, y0, x1, y1, w, wild = group_rect(t, dec(q0), dec(q1), W, H, slack_px, slack_w)
        for k in range(64):
            px, py, pw = project(t, dec(q[k]))
            ix = np.floor(fma((px / pw).astype(F), F(0.5), F(0.5)) * F(W))
            iy = np.floor(fma((py / pw).astype(F), F(0.5), F(0.5)) * F(H))
            ok = wild | ((ix >= x0) & (ix <= x1) & (iy >= y0) & (iy <= y1) & (pw >= w))
            assert ok.all()
    assert bounded >= 20


def layout(n, size, shift, shuffle):
    xyz, rgba = orc.generate(pcr.gen_cfg(pcr.SCENE_CITY, n, seed=size, num_buildings=9))
    if shuffle:
        perm = np.random.default_rng(size).permutation(n)
    else:
        perm = orc.morton_order(xyz)[0]
    b, lo, med, hi = pcr.encode_batches_host(xyz[perm], (size + 3) // 4 * 4)
    b["num_points"] = np.minimum(b["num_points"], size)   # the points behind belong to no batch
    rgba = rgba[perm]
    if not shift:
        return b, lo, med, hi, rgba
    out, src, pos, idx = b.copy(), [], 0, []
    for k in range(len(b)):   # 0..4 junk words in front of every batch
        gap, f, m = (k * 7 + 1) % 5, int(b[k]["first_point"]), int(b[k]["num_points"])
        idx.append(np.concatenate([np.zeros(gap, np.int64), np.arange(f, f + m)]))
        out[k]["first_point"] = pos + gap
        pos += gap + m
    idx = np.concatenate(idx)
    return out, lo[idx].copy(), med[idx].copy(), hi[idx].copy(), rgba[idx].copy()


def views():
    up = (0, 0, 1)
    yield pcr.look_at((150, -420, 260), (150, 150, 10), up=up, near=1, far=3000, width=333, height=211)
    yield pcr.look_at((60, 60, 25), (200, 200, 5), up=up, near=1, far=3000, width=1280, height=719)   # large, off the edges
    yield pcr.look_at((120, 120, 3), (121, 160, 2), up=up, near=0.01, far=3000, width=801, height=603)  # inside the cloud
    yield pcr.look_at((150, -9000, 6000), (150, 150, 0), up=up, near=1, far=30000, width=640, height=480)  # a few pixels


@pytest.mark.gpu
@pytest.mark.parametrize("n,size,shift,shuffle", [(70, 1, True, False), (1000, 63, True, False), (1000, 64, False, False),
                                                  (4003, 65, True, False), (9001, 1023, True, False),
                                                  (9001, 1024, False, False), (20011, 1025, True, False),
                                                  (150_001, 10240, True, False), (150_001, 16385, True, True),
                                                  (200_003, 200_003, True, False)])
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
def test_grouped_raster_equals_oracle(ctx, n, size, shift, shuffle, tile_px, block):
    b, lo, med, hi, rgba = layout(n, size, shift, shuffle)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    for v in views():
        ref, _ = orc.render_batched(b, lo, med, hi, v, 1)
        for skip in (True, False):
            fb = ctx.framebuffer(v.width, v.height)
            prm = pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block, occlusion_skip=skip)
            ctx.render(cloud, v, prm, fb)
            st = ctx.stats()
            assert np.array_equal(fb.keys(), ref), f"{v.width}x{v.height}: {(fb.keys() != ref).sum()} keys differ"
            assert st.points_occluded <= st.points_drawn and (skip or st.points_occluded == 0)
            # the same frame on top of itself: nearly every group is hidden
            ctx.render(cloud, v, pcr.params(pcr.MODE_LAS2, tile_px=tile_px, block_size=block, occlusion_skip=skip,
                                            clear_before=False), fb)
            assert np.array_equal(fb.keys(), ref) and ctx.stats().atomics_issued == 0
            fb.close()
        fb = ctx.framebuffer(v.width, v.height)
        ctx.render(cloud, v, pcr.params(pcr.MODE_LAS), fb)
        assert np.array_equal(fb.keys(), ref) and ctx.stats().points_occluded == 0
        fb.close()
    cloud.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,size,shift,shuffle", [(1000, 63, True, False), (20011, 1025, True, False),
                                                  (150_001, 10240, True, False), (150_001, 16385, True, True),
                                                  (200_003, 200_003, True, False)])
@pytest.mark.parametrize("tile_px,block", [(2048, 256), (1024, 128), (4096, 256)])
def test_grouped_hqs_equals_the_direct_passes(ctx, n, size, shift, shuffle, tile_px, block):
    """The direct passes (tile_px 0) are compared with the oracle elsewhere."""
    b, lo, med, hi, rgba = layout(n, size, shift, shuffle)
    cloud = ctx.upload_batched(b, lo, med, hi, rgba)
    for v in views():
        ref = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
        ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=0), ref)
        for skip in (True, False):
            fb = ctx.framebuffer(v.width, v.height, pcr.FB_HQS)
            ctx.render(cloud, v, pcr.params(pcr.MODE_HQS, tile_px=tile_px, block_size=block, occlusion_skip=skip), fb)
            st = ctx.stats()
            assert all(np.array_equal(a, r) for a, r in zip(fb.hqs(), ref.hqs()))
            assert st.points_occluded <= 2 * st.points_drawn and (skip or st.points_occluded == 0)
            fb.close()
        ref.close()
    cloud.close()
