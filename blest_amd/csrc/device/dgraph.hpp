// Host-side handles of the HBM-resident graph and of per-query device state.
#pragma once

#include <algorithm>
#include <atomic>

#include <hip/hip_runtime.h>

#include <functional>
#include <mutex>
#include <string>
#include <vector>

#include "../capi_internal.hpp"
#include "dev_common.hpp"
#include "segments.hpp"

namespace blest {

// The runtime keeps a failed call's error for the thread's next hipGetLastError, which is
// the check after a launch: taken here, so that the next call on the thread does not fail
// for what went wrong in this one.
#define BLEST_HIP(call)                                                                        \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) {                                                                \
            (void)hipGetLastError();                                                           \
            throw ::blest::Error(e_ == hipErrorOutOfMemory ? BLEST_ERR_OUT_OF_DEVICE_MEMORY    \
                                                           : BLEST_ERR_DEVICE,                 \
                                 std::string(#call) + ": " + hipGetErrorString(e_));           \
        }                                                                                      \
    } while (0)

// Read-only view of the device graph passed by value to kernels.
//
// HBM layout: the BVSS of the reference (sliceSetPtrs, virtualToReal, realPtrs, rowIds,
// masks) is uploaded with slice offsets converted to quad offsets: every vset holds a
// multiple of 4 slices (BVSS.cuh:379-415), so its slices are whole "quads" of 4 rows
// (one 16-byte uint4) and one 32-bit mask word (4 x 8-bit slice masks).  A wave64
// streams 64 quads = 256 slices per coalesced step (1 KiB of rows + 256 B of masks).
// Bitmaps (visited, frontier) are 64-bit words: word w holds vertices [64w, 64w+64),
// byte b of the bitmap is the frontier mask of real slice set b.
struct GraphView {
    uint32_t n, R, V, W;          // vertices, rsets, vsets, 64-bit bitmap words
    const uint32_t* unitQuad;     // V + 1: first quad of each vset
    const uint32_t* unitRset;     // V: owning rset (virtualToReal)
    const uint32_t* rsetUnit;     // R + 1: first vset of each rset (realPtrs)
    const uint4* rows;            // Q quads of row IDs (pad rows 0xFFFFFFFF)
    const uint32_t* masks;        // Q mask words
    const uint32_t* csrPtr;       // n + 1, bottom-up in-neighbour lists (nullable)
    const uint32_t* csrIdx;       // nnz
    const unsigned long long* noIn;  // W words: vertices without in-neighbours (nullable)
    const uint32_t* probe;        // n: each vertex's first in-neighbour (its highest-degree one:
                                  // the lists are sorted by degree); nullable
    unsigned long long nnz;       // directed edges
    const uint2* pullUnits;       // (vertex, first entry) of the list parts past kPullOwn entries
    uint32_t pullCount;
};

// Multi-source pull levels: a vertex's first kPullOwn list entries are scanned by the wave
// that owns its bitmap word, the rest in units of kPullUnit entries (pullUnits).
constexpr uint32_t kPullOwn = 64, kPullUnit = 256;

struct DeviceGraph {
    int device = 0;
    int cus = 0;
    uint32_t blockSize = 256, blocksPerCu = 4, gridBlocks = 0;
    // Producer segments of the single-source level kernels (one workgroup each), and the
    // wider set of the multi-source and label-propagation kernels, whose levels stream
    // records for long enough to want every workgroup slot.
    uint32_t segs = 1, wps = 1;    // segments and bitmap words per segment
    uint32_t* segBase = nullptr;   // segs + 1 first list slots
    uint32_t* chunkBase = nullptr; // segs + 1 first chunk slots (rsets of > kChunkVsets vsets)
    uint64_t chunks = 0;           // chunk slots in all
    uint32_t wideSegs = 1, wideWps = 1;
    uint32_t* wideBase = nullptr;  // wideSegs + 1 first list slots (no chunk lists)
    dev::SegView seg_view() const;
    dev::SegView wide_view() const;
    blest_device_opts opts{};
    uint32_t n = 0, R = 0, V = 0, W = 0;
    uint64_t S = 0, Q = 0, nnz = 0;
    bool symmetric = false, hasCsr = false, hasPerm = false;
    uint32_t *unitQuad = nullptr, *unitRset = nullptr, *rsetUnit = nullptr, *masks = nullptr;
    uint4* rows = nullptr;
    uint32_t *csrPtr = nullptr, *csrIdx = nullptr;
    unsigned long long* noIn = nullptr;  // bit v: v has no in-neighbour (never found bottom-up)
    uint32_t* probe = nullptr;           // first bottom-up probe per vertex
    uint2* pullUnits = nullptr;
    uint32_t pullCount = 0;
    bool thin = false;                   // short lists: single-source levels over vertex queues
    bool small = false;                  // few vertices and edges: one workgroup's BFS, unless thin
    // a queue traversal of this graph had few, wide levels: the bit-matrix levels are faster
    // (the graph's, not a query's: queries are made anew, and blest_bfs_noalloc has none)
    std::atomic<bool> thinWide{false};
    // what blest_bfs_noalloc keeps from one traversal of this graph to the next (under the
    // lock of its device's scratch)
    unsigned noallocHint = 0;
    bool noallocOnQueues = false;
    uint32_t thinSegs = 1, thinShift = 0;
    size_t thin_queue_entries() const { return size_t(thinSegs) << (6 + thinShift); }
    uint32_t *permNewToOld = nullptr, *permOldToNew = nullptr;  // device copies
    std::vector<uint32_t> hostOldToNew, hostNewToOld;
    std::vector<uint32_t> hostDegree;  // per (reordered) vertex, for GTEPS accounting
    uint64_t deviceBytes = 0;
    std::vector<void*> allocations;

    GraphView view() const {
        GraphView g;
        g.n = n;
        g.R = R;
        g.V = V;
        g.W = W;
        g.unitQuad = unitQuad;
        g.unitRset = unitRset;
        g.rsetUnit = rsetUnit;
        g.rows = rows;
        g.masks = masks;
        g.csrPtr = csrPtr;
        g.csrIdx = csrIdx;
        g.noIn = noIn;
        g.probe = probe;
        g.nnz = nnz;
        g.pullUnits = pullUnits;
        g.pullCount = pullCount;
        return g;
    }
    template <class T>
    T* alloc(size_t count) {
        void* p = nullptr;
        BLEST_HIP(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)));
        allocations.push_back(p);
        deviceBytes += count * sizeof(T);
        return static_cast<T*>(p);
    }
    ~DeviceGraph();
};

// A captured chunk of levels (kernels that read their level from ctrl->levelBase),
// replayed until the traversal finishes.  key = the launch parameters it was captured
// with; a different key recaptures.
struct LevelGraph {
    hipGraphExec_t exec = nullptr;
    unsigned chunk = 0;
    uint64_t key = 0;
};
enum LevelGraphKind { kGraphBfs = 0, kGraphMbfs1 = 1, kGraphMbfs2 = 2, kGraphThin = 3, kGraphCount = 4 };
constexpr unsigned kGraphChunkLevels = 16;  // levels per replayed graph
constexpr unsigned kGraphMinLevels = 64;    // auto mode: replay once a traversal was this deep

// Mutable per-query device state.
struct Query {
    DeviceGraph* g = nullptr;
    uint32_t maxSources = 1;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipEvent_t evIn = nullptr;     // a caller's stream position that the next launch waits for
    // pinned: a chunk's closing kernel stores the control block here, so a poll is one
    // stream synchronisation (no copy, no second round trip for the totals)
    dev::Ctrl* hostCtrl = nullptr;
    int32_t* hostStage = nullptr;  // pinned, kStageBytes at most, made for the first small host result
    size_t hostStageCount = 0;
    unsigned headSkip = 0;         // traversals to go without the fused kernel right after the init
                                   // kernel, since the last one found no level to run there
    unsigned levelHint = 0;        // levels of the last traversal (sizes the first chunk)
    dev::Ctrl* ctrl = nullptr;
    int32_t* levels = nullptr;  // n * maxSources
    unsigned long long *visited = nullptr, *front0 = nullptr, *front1 = nullptr, *next = nullptr;
    uint8_t* nextB = nullptr;  // single-source top-down discoveries, a byte per vertex (W * 64)
    uint32_t *list0 = nullptr, *list1 = nullptr;
    uint2 *chunk0 = nullptr, *chunk1 = nullptr;        // chunk lists (single-source BFS)
    uint32_t *segCount = nullptr, *segNew = nullptr;  // [3][segments]
    uint32_t* segChunks = nullptr;                     // [3][segments]
    unsigned long long* segEdges = nullptr;            // [3][segments]
    dev::SegCounters seg_counters() const;
    // vertex queues of a thin graph's levels (thin_levels.hpp); null otherwise
    uint32_t *thinQueue0 = nullptr, *thinQueue1 = nullptr, *thinCount = nullptr;
    unsigned long long* thinEdges = nullptr;
    bool onQueues = false;  // the last single-source traversal ran on them (levelHint counts its levels)
    int32_t* levelsOut = nullptr;  // original-order copy (when the graph carries a permutation)
    uint32_t* labels = nullptr;    // CC
    uint32_t* labelsAux = nullptr;
    uint32_t* ccCounts = nullptr;  // per workgroup: roots, the giant tree's minimum; then its root as voted and in the end
    std::vector<uint32_t> hostCcCounts;
    // multi-source state, allocated on first use: words per vertex x n
    uint32_t mbfsWords = 0;
    unsigned long long *mVis = nullptr, *mFront0 = nullptr, *mFront1 = nullptr, *mNext = nullptr;
    unsigned long long* mHist = nullptr;  // frontier words of levels 0..mHistLevels
    unsigned long long* mFull = nullptr;  // rows every root has reached (1 bit per vertex)
    unsigned long long* mAny = nullptr;   // 2 x W: vertices in the frontier of some root (1 bit), by level parity
    uint8_t* mDirty = nullptr;            // W: words whose `next` words were set in the running level
    uint32_t mHistLevels = 0;
    void* rootStats = nullptr;  // per-root totals of a multi-source run, 128 entries
    LevelGraph graphs[kGraphCount];
    bool noGraphs = false;  // never replay captured level chunks (queries of the request server)
    std::vector<hipEvent_t> traceEvents;  // one per traced kernel boundary (created on demand)
    std::vector<void*> allocations;
    std::mutex mu;
    uint32_t lastSource = 0;
    bool pending = false;

    template <class T>
    T* alloc(size_t count) {
        void* p = nullptr;
        BLEST_HIP(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)));
        allocations.push_back(p);
        return static_cast<T*>(p);
    }
    void release(void* p) {
        if (!p) return;
        auto it = std::find(allocations.begin(), allocations.end(), p);
        if (it == allocations.end()) return;
        (void)hipStreamSynchronize(stream);
        (void)hipFree(p);
        allocations.erase(it);
    }
    ~Query();
};

// Lays a single-source traversal's state over `base` (256-byte aligned pieces; the level
// array too when asked for, the vertex queues of a thin graph, the bitmap of the
// label-propagation components) and returns the bytes it takes.  With base == nullptr it
// only measures.
size_t carve_state(const DeviceGraph& g, unsigned char* base, Query& q, bool withLevels, bool thin, bool withNext);

// Level-loop driver: enqueues level(L) for L = 1, 2, ... in chunks and polls the
// device's done flag after each chunk.  tail (nullable) enqueues the traversal's closing
// kernel after each chunk: it stores the control block in q.hostCtrl and does its work
// only once the traversal is done; ev1 is recorded after it.  With lg and levelRel given (levelRel(k) launches
// level levelBase + k), deep traversals replay a captured chunk of levels instead
// (device opts use_graphs: 0 auto, 1 always, 2 never; queries with noGraphs never).
dim3 level_grid(const DeviceGraph& g);
dim3 wide_grid(const DeviceGraph& g);
// after / afterRel (nullable): a kernel enqueued after each chunk of levels, given the
// next level (absolute / relative to the replayed chunk); with it the first chunk is the
// previous traversal's levelHint levels instead of levelHint + 2.
void run_levels(Query& q, const std::function<void(unsigned)>& level, const std::function<void()>& tail = nullptr,
                LevelGraph* lg = nullptr, const std::function<void(unsigned)>& levelRel = nullptr,
                uint64_t key = 0, const std::function<void(unsigned)>& after = nullptr,
                const std::function<void(unsigned)>& afterRel = nullptr);
uint64_t launch_key(double alpha, double beta, int direction, uint64_t extra);
uint32_t map_source(const DeviceGraph& g, uint32_t src);
// Levels of multi-source frontier words kept for the final level expansion: up to 16,
// within 32 GiB of history per query.
inline uint32_t mbfs_history_levels(uint32_t n, uint32_t nw) {
    const uint64_t perLevel = uint64_t(n) * nw * 8;
    const uint64_t fit = (uint64_t(32) << 30) / std::max<uint64_t>(perLevel, 1);
    return uint32_t(std::min<uint64_t>(16, std::max<uint64_t>(fit, 2) - 1));
}
// Result destinations.  A caller's array may be host memory or device memory of the
// graph's device; when it is device memory, [dst, dst + bytes) must lie inside one
// allocation (hipMemGetAddressRange), else BLEST_ERR_INVALID_ARGUMENT is thrown before
// anything is copied: an undersized or wrong-graph buffer becomes an error, not an
// out-of-bounds device write.  Host memory cannot be measured and is taken as given.
// Returns whether dst is device memory.
bool check_result_range(const void* dst, size_t bytes, int device, const char* what);
// trace (nullable): record an event after the init kernel and after every level kernel.
// dst (nullable): the caller's device array (original order), written by the closing kernel.
void bfs_launch(Query& q, uint32_t srcReordered, bool trace = false, int32_t* dst = nullptr);
void bfs_finish(Query& q, int32_t* hostLevels, blest_bfs_stats* st);
// Where a traversal may write n x rows results directly: dst when it is device memory
// (checked to fit) apart from the query's own level array, else null.
// onHost (nullable): whether dst is host memory.
int32_t* direct_result(const Query& q, int32_t* dst, size_t count, const char* what, bool* onHost = nullptr);
// Small results for host memory are written by the closing kernel into pinned memory of the
// query and copied from there: the runtime's copy to pageable memory is a staging copy of
// its own with a second wait.  A traversal with a host result: 65.9 -> 41.5 us at 16 KB,
// 139.9 -> 125.0 at 256 KB, 181.1 -> 170.8 at 1 MB; no gain from 2 MB on, where the copy
// engine is the faster way out.  Null: too large, or no pinned memory to be had.
constexpr size_t kStageBytes = size_t(1) << 20;
int32_t* host_stage(Query& q, size_t count);

}  // namespace blest

struct blest_device_graph {
    blest::DeviceGraph g;
};
struct blest_query {
    blest::Query q;
};
