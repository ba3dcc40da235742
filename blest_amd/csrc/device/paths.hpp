// Which symmetric graphs with a resident CSR have their single-source BFS on kernels of their
// own: one workgroup, or vertex queues.  (No HIP in here: the host test compiles it as it is.)
#pragma once

#include <stdint.h>

namespace blest {
namespace dev {

// Graphs traversed over vertex queues (thin_levels.hpp): at most kThinMeanDegree list
// entries a vertex on average, and
//   no list longer than kThinMaxDegree (grids, road networks: many levels), up to
//     kThinMaxVertices, past which a level's claims outweigh what its launches save (us per
//     BFS, queues and bit matrix: grids of 300, 1000, 2047 and 4096 squared 314 and 585,
//     489 and 917, 812 and 1602, 4532 and 3373);
//   or no list longer than kThinMidDegree (sparse random graphs) from kThinMidFrom
//     vertices, below which one workgroup is faster (bfs_small_kernel; mean degree 4: 8 K
//     vertices 78 against 90, 20 K 149 against 114), up to kThinMidEdges (mean degree 3:
//     0.1 M vertices 144 and 219, 0.26 M 200 and 275, 0.4 M 227 and 296, 0.8 M 339 and 313).
// A graph that passes but turns out to have few, wide levels (kThinFewLevels,
// kThinWideLevel vertices on average) is left to the bit matrix after its first traversal.
constexpr uint32_t kThinMeanDegree = 5, kThinMaxDegree = 8, kThinMidDegree = 32;
constexpr uint32_t kThinMaxVertices = 6u << 20, kThinMidFrom = 8192, kThinMidEdges = 21u << 16;
constexpr uint32_t kThinFewLevels = 40, kThinWideLevel = 32768;

constexpr bool thin_graph(uint32_t n, uint64_t nnz, uint32_t maxDegree) {
    return nnz <= uint64_t(kThinMeanDegree) * n &&
           (maxDegree <= kThinMaxDegree ? n <= kThinMaxVertices
                                        : maxDegree <= kThinMidDegree && n > kThinMidFrom && nnz <= kThinMidEdges);
}

// Graphs that one workgroup (bfs_small_kernel) traverses faster than level kernels do.  Its
// time grows with the words of the bitmap, which every level passes over, and with the edges;
// a level pair costs 15 us and more whatever it holds (us per call, one workgroup and level
// kernels: Erdos-Renyi of mean degree 4, 2 K vertices 44 and 139, 8 K 78 and 142, 20 K 149
// and 177; mean degree 3, 50 K 397 and 224; R-MAT 13 of edge factor 16 52 and 104).
constexpr uint32_t kSmallVertices = 16384, kSmallEdges = 1u << 18;
constexpr bool small_graph(uint32_t n, uint64_t nnz) { return n <= kSmallVertices && nnz <= kSmallEdges; }

}  // namespace dev
}  // namespace blest
