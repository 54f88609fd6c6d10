"""The per-frame counters: each workgroup adds what it counted to one of
several slots in lines of their own, and pcr_stats adds the slots."""
import os
import subprocess

import numpy as np
import pytest

import compute_rasterizer_amd as pcr
from oracle import orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

LAYOUT = r"""
#include <cstddef>
#include "pcr_internal.h"
using namespace pcr;
// the counters that every workgroup adds to share no line with the work queue or with another slot's
static_assert(sizeof(FrameCounts) >= 128 && alignof(FrameCounts) >= 128, "slot");
static_assert(offsetof(FrameState, counts) >= 128 && sizeof(FrameState::counts) == kCountSlots * sizeof(FrameCounts), "state");
static_assert(kCountSlots >= 16, "slots");   // 1,536 workgroups, 4 atomics of 12 ns: under 5 us a slot
int main() {}
"""


def test_counters_have_lines_of_their_own(tmp_path):
    src = tmp_path / "layout.cpp"
    src.write_text(LAYOUT)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "compute_rasterizer_amd", "csrc"), str(src)], check=True)


@pytest.mark.gpu
@pytest.mark.parametrize("per_batch", [1, 4, 64])
def test_every_workgroup_is_counted(ctx, per_batch):
    """Points on pixels of their own: a frame issues one atomic a point, and
    the same frame on top of itself none."""
    u, v = np.meshgrid(np.arange(80), np.arange(60), indexing="ij")
    xyz = np.stack([(u * 8 + 4.5) / 320.0 - 1.0, (v * 8 + 4.5) / 240.0 - 1.0, np.zeros(u.shape)], -1)
    xyz = xyz.reshape(-1, 3).astype(np.float32) * np.array([640 / 480, 1.0, 1.0], np.float32)
    b, lo, med, hi = pcr.encode_batches_host(xyz, max(4, per_batch))
    b["num_points"] = np.minimum(b["num_points"], per_batch)   # the points behind belong to no batch
    view = pcr.look_at((0, 0, 1.75), (0, 0, 0), up=(0, 1, 0), near=0.1, far=100, width=640, height=480)
    ref, _ = orc.render_batched(b, lo, med, hi, view, 1)
    n = int(b["num_points"].sum())
    assert (ref != np.uint64(0xFFFFFFFFFFFFFFFF)).sum() == n and len(b) >= 64
    cloud = ctx.upload_batched(b, lo, med, hi, np.arange(len(xyz), dtype=np.uint32))
    for prm in (dict(mode=pcr.MODE_LAS2), dict(mode=pcr.MODE_LAS2, tile_px=0), dict(mode=pcr.MODE_LAS),
                dict(mode=pcr.MODE_LAS, block_size=64)):
        fb = ctx.framebuffer(640, 480)
        for _ in range(3):   # the two frame states in turn
            ctx.render(cloud, view, pcr.params(**prm), fb)
            assert np.array_equal(fb.keys(), ref) and ctx.stats().atomics_issued == n
        ctx.render(cloud, view, pcr.params(clear_before=False, **prm), fb)
        assert np.array_equal(fb.keys(), ref) and ctx.stats().atomics_issued == 0
        fb.close()
    cloud.close()
