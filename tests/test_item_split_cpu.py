"""CPU: how a launch's workgroups share out the listed batches (ItemSplit) and
cut a batch into parts (batch_part), as the kernels compile them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "pcr_internal.h"
using namespace pcr;
#define REQUIRE(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

static void items(uint32_t count, uint32_t groups) {
    ItemSplit w;
    w.split(count, groups);
    std::vector<uint32_t> seen(count, 0), parts_of(count, 0);
    uint32_t last_part = 0;
    for (uint32_t i = 0; i < w.items; i++) {
        uint32_t part, parts;
        const uint32_t b = w.batch_of(i, part, parts);
        REQUIRE(b < count && part < parts && parts <= kMaxParts);
        REQUIRE((seen[b] & (1u << part)) == 0);
        REQUIRE(parts_of[b] == 0 || parts_of[b] == parts);
        REQUIRE(parts == 1 || part >= last_part);   // all first parts, then all second ones
        if (parts > 1) last_part = part;
        seen[b] |= 1u << part;
        parts_of[b] = parts;
    }
    for (uint32_t b = 0; b < count; b++) REQUIRE(seen[b] == (1u << parts_of[b]) - 1u);
    // a short list gives most of the workgroups an item of its own
    const uint64_t can = (uint64_t)count * kMaxParts < groups ? (uint64_t)count * kMaxParts : groups;
    REQUIRE(2 * (uint64_t)w.items >= can);
}

static void cut(uint32_t first, uint32_t np, uint32_t parts) {
    uint32_t next = first;
    for (uint32_t p = 0; p < parts; p++) {
        pcr_batch h{};
        h.first_point = first;
        h.num_points = np;
        batch_part(h, p, parts);
        REQUIRE(part_empty(first, np, p, parts) == (h.num_points == 0));
        if (h.num_points == 0) continue;
        REQUIRE(h.first_point == next);                                          // in order, none left out
        REQUIRE(p == 0 || (h.first_point - (first & ~3u)) % kPartRound == 0);   // whole rounds and groups
        next = h.first_point + h.num_points;
    }
    REQUIRE(next == first + np);
}

int main() {
    for (uint32_t groups : {1u, 2u, 30u, 1024u, 1536u, 2048u})
        for (uint32_t count : {0u, 1u, 2u, 3u, 10u, 97u, 98u, 511u, 512u, 767u, 768u, 1024u, 1535u, 1536u, 5000u})
            items(count, groups);
    for (uint32_t first : {0u, 1u, 2u, 3u, 10243u, 4000000000u})
        for (uint32_t np : {0u, 1u, 63u, 1021u, 1022u, 1023u, 1024u, 1025u, 2047u, 2048u, 2049u, 10240u, 16385u, 200003u, 100000000u})
            for (uint32_t parts = 2; parts <= kMaxParts; parts++) cut(first, np, parts);
    // both halves of a batch of one round: one has nothing to draw
    REQUIRE(!part_empty(0, 1024, 0, 2) && part_empty(0, 1024, 1, 2));
}
"""


def test_items_and_parts(tmp_path):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "compute_rasterizer_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


ROUNDS = r"""
#include <cstdio>
#include "pcr_internal.h"
using namespace pcr;
int main() {
    // between half the workgroups and all of them: halves of 977 batches on
    // 1,536 workgroups end after a whole batch's time, thirds after two thirds
    for (uint32_t groups : {1024u, 1536u, 2048u})
        for (uint32_t count = groups / 2 + 1; count < groups; count++) {
            ItemSplit w;
            w.split(count, groups);
            for (uint32_t p = 2; p <= 4; p++) {
                const uint32_t mine = (count * w.nparts + groups - 1) / groups, other = (count * p + groups - 1) / groups;
                if ((uint64_t)mine * p > (uint64_t)other * w.nparts) {
                    std::printf("%u batches, %u workgroups: %u parts, %u better\n", count, groups, w.nparts, p);
                    return 1;
                }
            }
        }
}
"""


def test_lists_near_the_number_of_workgroups(tmp_path):
    src, exe = tmp_path / "rounds.cpp", tmp_path / "rounds"
    src.write_text(ROUNDS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "compute_rasterizer_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
