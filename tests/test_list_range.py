"""Walks of adjacency lists next to entry 2^32 of the list array (CPU): the position helpers
that the traversal kernels use (csrc/device/list_range.hpp, compiled as it is), in the shapes
the kernels walk lists in: every entry exactly once, and an end."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "device/list_range.hpp"
using namespace blest::dev;

static int failures = 0;
static void check(const std::vector<unsigned>& seen, uint32_t begin, uint32_t end, const char* what) {
    bool ok = seen.size() == end - begin;
    for (unsigned s : seen) ok = ok && s == 1;
    if (!ok && ++failures < 20) std::printf("%s: list [%u, %u)\n", what, begin, end);
}

int main() {
    const uint64_t top = uint64_t(1) << 32;
    for (uint32_t len : {0u, 1u, 3u, 4u, 15u, 16u, 63u, 64u, 65u, 255u, 256u, 257u, 321u, 700u})
        for (uint32_t below : {1u, 2u, 3u, 4u, 15u, 16u, 17u, 63u, 64u, 65u, 255u, 256u, 1000u}) {
            const uint32_t end = uint32_t(top - below), begin = end - len;
            std::vector<unsigned> seen(len, 0);
            const auto hit = [&](uint32_t p) {
                if (p - begin < len) ++seen[p - begin];
                else ++failures;
            };
            const auto next = [&](const char* what) {
                check(seen, begin, end, what);
                seen.assign(len, 0);
            };
            // a lane: 2, then 4 entries a step
            for (uint32_t p = begin, step = 2; p < end; step = 4) {
                const uint32_t len = step < end - p ? step : end - p;
                for (uint32_t i = 0; i < 4; ++i)
                    if (i < len) hit(p + i);
                p += len;
            }
            next("lane steps");
            // a wave: 64 entries a step
            unsigned steps = 0;
            for (uint32_t q0 = begin; q0 < end && ++steps < 100; q0 = part_end(q0, end, 64))
                for (uint32_t lane = 0; lane < 64; ++lane)
                    if (in_part(q0, lane, end)) hit(q0 + lane);
            next("wave steps");
            // a row of 16 lanes up to 64 entries, the rest in units of 256, 4 entries a lane
            const uint32_t own = part_end(begin, end, 64);
            for (uint32_t s = 0; s < 64; s += 16)
                for (uint32_t sub = 0; sub < 16; ++sub)
                    if (in_part(begin, s, own) && in_part(begin, s + sub, own)) hit(begin + s + sub);
            for (uint32_t p0 = own; p0 < end; p0 = part_end(p0, end, 256)) {
                const uint32_t p1 = part_end(p0, end, 256);
                for (uint32_t lane = 0; lane < 64; ++lane)
                    for (uint32_t j = 0; j < 4; ++j)
                        if (in_part(p0, lane * 4, p1) && in_part(p0, lane * 4 + j, p1)) hit(p0 + lane * 4 + j);
            }
            next("row and units");
            // the first entries, the next ones, the rest a wave apart
            const uint32_t first = part_end(begin, end, 1), last = part_end(begin, end, 3);
            for (uint32_t i = begin; i < first; ++i) hit(i);
            for (uint32_t i = first; i < last; ++i) hit(i);
            for (uint32_t lane = 0; lane < 64; ++lane)
                for (uint32_t i = lane; in_part(last, i, end); i += 64) hit(last + i);
            next("samples and rest");
        }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
"""


def test_walks_at_the_end_of_the_index_range(tmp_path):
    src, exe = tmp_path / "walks.cpp", tmp_path / "walks"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", f"-I{ROOT / 'blest_amd' / 'csrc'}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_kernels_keep_to_the_helpers():
    """No walk over the list array compares a sum of a position and a step."""
    import re
    dev = ROOT / "blest_amd" / "csrc" / "device"
    sums = re.compile(r"min\([^()]*, *(p|q0|p0|b|hb) \+ \w+\)|\bmin\((p|q0|p0|b|hb) \+ |"
                      r"\b(q0|hb|p0|p) \+ \w+ < (q1|p1|e|he|lim)\b")
    for name in ("bfs.hip", "mbfs.hip", "cc.hip"):
        found = [l.strip() for l in (dev / name).read_text().splitlines() if sums.search(l)]
        assert not found, (name, found)
