"""Which graphs leave the single-source level kernels (CPU): the rules of csrc/device/paths.hpp,
compiled as they are, on both sides of every bound."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

# vertices, list entries, longest list -> vertex queues, one workgroup (which comes second)
CASES = [
    (1, 0, 0, True, True),
    (2003, 16024, 21, False, True),
    (16384, 262144, 300, False, True),      # both bounds of the one-workgroup path
    (16384, 262145, 300, False, False),
    (16385, 100000, 300, False, False),
    (16384, 5 * 16384, 8, True, True),      # five entries a vertex
    (16384, 5 * 16384 + 1, 8, False, True),
    (6 << 20, 20 << 20, 8, True, False),    # vertices of a short-list graph
    ((6 << 20) + 1, 20 << 20, 8, False, False),
    (8192, 30000, 9, False, True),          # medium lists: vertices, length, entries
    (8193, 30000, 9, True, True),
    (300000, 1376256, 32, True, False),
    (300000, 1376256, 33, False, False),
    (300000, 1376257, 32, False, False),
    (300000, 1376257, 8, True, False),
]

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "device/paths.hpp"
int main(int, char** v) {
    const uint32_t n = std::strtoul(v[1], 0, 10), longest = std::strtoul(v[3], 0, 10);
    const uint64_t nnz = std::strtoull(v[2], 0, 10);
    std::printf("%d %d\n", int(blest::dev::thin_graph(n, nnz, longest)), int(blest::dev::small_graph(n, nnz)));
}
"""


def test_path_bounds(tmp_path):
    src, exe = tmp_path / "paths.cpp", tmp_path / "paths"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", f"-I{ROOT / 'blest_amd' / 'csrc'}", str(src), "-o", str(exe)],
                   check=True)
    for n, nnz, longest, queues, small in CASES:
        got = subprocess.run([str(exe), str(n), str(nnz), str(longest)], capture_output=True, text=True, check=True)
        assert got.stdout.split() == [str(int(queues)), str(int(small))], (n, nnz, longest)
