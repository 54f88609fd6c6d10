"""CPU: group_rect(), compiled for the host from the kernels' header, holds the
points of its group at every precision level: at the 20- and 30-bit levels the
box holds the upper 10 bits of a coordinate and is open upwards by one step.

The host stands in for one instruction: v_rcp_f32 is within 1 ulp, so the
reciprocal is tried exactly rounded, one step up and one step down."""
import os
import subprocess

import numpy as np
import pytest

import compute_rasterizer_amd as pcr

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __restrict__
using std::max;
using std::min;
struct uint2 { uint32_t x, y; };
struct Decode { float scale[3], mn[3]; };
static int g_ulp = 0;
static float fma_(float a, float b, float c) { return std::fma(a, b, c); }
static float rcp(float x) {
    const float r = 1.0f / x;
    return g_ulp == 0 ? r : std::nextafterf(r, g_ulp > 0 ? INFINITY : -INFINITY);
}
#define __builtin_amdgcn_rcpf rcp
"""

PROGRAM = r"""
struct Case { float t[16], mn[3], mx[3]; int32_t w, h; };
// decode() of the header at one level, from a coordinate's 30 bits
static float coord(int level, uint32_t X, const Decode& d, int a) {
    const uint32_t v = level == 0 ? X : level == 1 ? X & ~1023u : X >> 20;
    return fma_((float)v, d.scale[a], d.mn[a]);
}
int main(int argc, char** argv) {
    std::vector<Case> cases;
    std::FILE* f = std::fopen(argv[1], "rb");
    for (Case c; std::fread(&c, sizeof c, 1, f) == 1;) cases.push_back(c);
    std::fclose(f);
    std::mt19937 rng(12345);
    long bounded[3] = {0, 0, 0}, tight[3] = {0, 0, 0}, points = 0;
    for (const Case& c : cases)
        for (int level = 0; level <= 2; level++) {
            const float* t = c.t;
            Decode d;
            for (int a = 0; a < 3; a++) {
                d.scale[a] = (c.mx[a] - c.mn[a]) * (level <= 1 ? 0x1p-30f : 0x1p-10f);
                d.mn[a] = c.mn[a];
            }
            // screen_rect()'s wnear
            float pwmin = INFINITY, e[3];
            for (int k = 0; k < 8; k++)
                pwmin = std::min(pwmin, fma_(t[11], (k & 4 ? c.mx : c.mn)[2],
                                             fma_(t[7], (k & 2 ? c.mx : c.mn)[1], fma_(t[3], (k & 1 ? c.mx : c.mn)[0], t[15]))));
            const int row[3] = {0, 1, 3};
            for (int r = 0; r < 3; r++) {
                e[r] = std::fabs(t[12 + row[r]]);
                for (int a = 0; a < 3; a++) e[r] += std::fabs(t[4 * a + row[r]]) * std::max(std::fabs(c.mn[a]), std::fabs(c.mx[a]));
            }
            const float side = (float)std::max(c.w, c.h);
            if (!(pwmin >= 0x1p-12f + 0x1p-16f * e[2] && pwmin >= side * 0x1p-21f * (std::max(e[0], e[1]) + e[2]))) continue;
            const float wnear = pwmin - 0x1p-18f * e[2];
            if (!(wnear > 0)) continue;
            const GroupSlack s = group_slack(t, c.mn, c.mx, c.w, c.h, wnear);
            for (int g = 0; g < 300; g++) {
                uint32_t lo[3], hi[3], bits[3][64];
                const int span = 1 + (int)(rng() % (g % 3 == 0 ? 2 : g % 3 == 1 ? 16 : 200));
                uint2 box{0, 0};
                for (int a = 0; a < 3; a++) {
                    lo[a] = rng() % 1024;
                    hi[a] = std::min(lo[a] + (uint32_t)(rng() % span), 1023u);
                    for (int k = 0; k < 64; k++) {
                        // the ends of the box, and points next to its faces, among them
                        const uint32_t l = k == 0 ? lo[a] : k == 1 ? hi[a] : lo[a] + (uint32_t)(rng() % (hi[a] - lo[a] + 1));
                        const uint32_t sub = k % 4 == 0 ? 0u : k % 4 == 1 ? 0xFFFFFu : (uint32_t)(rng() & 0xFFFFFu);
                        bits[a][k] = l << 20 | sub;
                    }
                    box.x |= lo[a] << (10 * a);
                    box.y |= hi[a] << (10 * a);
                }
                for (g_ulp = -1; g_ulp <= 1; g_ulp++) {
                    const GroupRect r = group_rect(box, level, d, t, c.w, c.h, s.px, s.w);
                    if (r.wild) continue;
                    bounded[level]++;
                    tight[level] += (r.x1 - r.x0) * (r.y1 - r.y0) < 4096;
                    for (int k = 0; k < 64; k++) {
                        const float x = coord(level, bits[0][k], d, 0), y = coord(level, bits[1][k], d, 1), z = coord(level, bits[2][k], d, 2);
                        const float px = fma_(t[8], z, fma_(t[4], y, fma_(t[0], x, t[12]))),
                                    py = fma_(t[9], z, fma_(t[5], y, fma_(t[1], x, t[13]))),
                                    pw = fma_(t[11], z, fma_(t[7], y, fma_(t[3], x, t[15])));
                        points++;
                        if (!(pw >= r.w)) { std::printf("level %d: depth %.9g below %.9g\n", level, pw, r.w); return 1; }
                        const float nx = px / pw, ny = py / pw;
                        if (!(nx >= -1 && nx <= 1 && ny >= -1 && ny <= 1)) continue;
                        const int ix = (int)(fma_(nx, 0.5f, 0.5f) * (float)c.w), iy = (int)(fma_(ny, 0.5f, 0.5f) * (float)c.h);
                        if (ix >= c.w || iy >= c.h) continue;
                        if (ix < r.x0 || ix > r.x1 || iy < r.y0 || iy > r.y1) {
                            std::printf("level %d: pixel %d %d outside %d..%d %d..%d\n", level, ix, iy, r.x0, r.x1, r.y0, r.y1);
                            return 1;
                        }
                    }
                }
            }
        }
    std::printf("%ld %ld %ld bounded, %ld %ld %ld tight, %ld points\n", bounded[0], bounded[1], bounded[2], tight[0], tight[1], tight[2], points);
    return 0;
}
"""


@pytest.mark.parametrize("offset,extent", [(0.0, 100.0), (5000.0, 40.0), (-2000.0, 30.0), (1.0e5, 500.0)])
def test_group_rect_holds_its_points_at_every_level(tmp_path, offset, extent):
    with open(os.path.join(ROOT, "compute_rasterizer_amd", "csrc", "pcr_device.h")) as f:
        header = f.read()
    body = header[header.index("struct GroupSlack {"):header.index("// A batch's screen rectangle for one view")]
    rng = np.random.default_rng(int(extent))
    cases = []
    for k in range(60):
        mn = (offset + rng.uniform(-extent, extent, 3)).astype(np.float32)
        mx = (mn + rng.uniform(0.01, extent, 3).astype(np.float32)).astype(np.float32)
        mid = 0.5 * (mn + mx)
        eye = mid + rng.normal(size=3) * extent * rng.uniform(0.5, 6)
        w, h = int(rng.integers(3, 4000)), int(rng.integers(3, 3000))
        v = pcr.look_at(tuple(map(float, eye)), tuple(map(float, mid + rng.normal(size=3) * extent * 0.3)), up=(0, 0, 1),
                        near=0.01, far=1e6, width=w, height=h)
        cases.append(np.array(v.transform[:], np.float32).tobytes() + mn.tobytes() + mx.tobytes() + np.array([w, h], np.int32).tobytes())
    data, src, exe = tmp_path / "cases", tmp_path / "bound.cpp", tmp_path / "bound"
    data.write_bytes(b"".join(cases))
    src.write_text(PRELUDE + body + PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-mfma", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe), str(data)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    bounded, tight = (list(map(int, p.split()[:3])) for p in out.stdout.split(",")[:2])
    assert min(bounded) > 10_000 and min(tight) > 1000, out.stdout
