// Top-down BFS levels over vertex queues, for graphs whose lists are short (grids, road
// networks, sparse random graphs; paths.hpp): symmetric, resident CSR, few entries a vertex
// on average.  Such a traversal has dozens of thin levels.  In the bit-matrix form a
// level is two kernels, and both touch every segment whatever the frontier holds: the
// update packs a byte per vertex, the expansion looks up a vset and a frontier byte per
// listed rset.  Bottom-up sweeps do not pay either: a list of four seldom ends early.  Here
// a level is one kernel: a thread takes a frontier vertex, claims its unvisited neighbours
// with an atomicOr on the visited bitmap (no two hubs meet in one word) and appends them to
// the next queue.
//
// The queue is segmented by vertex ID: segment s holds the vertices of bitmap words
// [s << shift, (s + 1) << shift), so its room, 64 << shift entries, bounds what a level can
// append to it and no append can overflow.  Counters rotate over three slots: level L reads
// slot L % 3, appends to slot (L + 1) % 3 and clears slot (L + 2) % 3.
//
// Bound by the chain of dependent round trips of a level (counters, queue entry, list
// bounds, list, visited word, claim, append), not by bandwidth.  Measured (MI355X),
// 2047-square grid in RCM order, ~70 levels: 1.56 -> 0.91 ms per traversal (18 + 10 us a
// level before, 10 us at 2 K frontier vertices, 38 us at 330 K: claims at about 12 G/s).
#pragma once

#include "level_common.hpp"
#include "paths.hpp"
#include "small_traverse.hpp"

namespace blest {
namespace dev {

constexpr int kThinBlock = 512;
constexpr int kThinFusedBlock = 1024;
constexpr uint32_t kThinCap = 4096;      // queue entries a one-workgroup level may hold
constexpr uint32_t kThinEnter = 2048;    // entries with which a growing frontier stays there

struct ThinArgs {
    int32_t* levels;
    uint32_t* visited;               // 32-bit view of the bitmap
    uint32_t *queue0, *queue1;       // by level parity
    uint32_t* count;                 // [3][kThinMaxSegs]
    unsigned long long* edges;       // [kThinMaxSegs]: degree sum by workgroup
    Ctrl* ctrl;
    uint32_t segs, shift;            // shift: log2 of a segment's bitmap words
    uint32_t src;
    int levelFromCtrl;
};

__global__ void __launch_bounds__(kProducerBlock) thin_init_kernel(GraphView g, ThinArgs a) {
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x, nthreads = gridDim.x * blockDim.x;
    for (uint32_t w = tid; w < g.W * 2; w += nthreads) a.visited[w] = w == a.src >> 5 ? 1u << (a.src & 31) : 0u;
    const uint32_t seg = a.src >> (6 + a.shift);
    for (uint32_t i = tid; i < 3 * kThinMaxSegs; i += nthreads) a.count[i] = i == kThinMaxSegs + seg ? 1u : 0u;
    for (uint32_t i = tid; i < kThinMaxSegs; i += nthreads) a.edges[i] = 0ull;
    if (tid == 0) {
        a.queue1[seg << (6 + a.shift)] = a.src;  // level 1 reads the odd queue
        a.levels[a.src] = 0;
        level_state_reset(a.ctrl);
    }
}

// What level L reads: the inclusive prefix of its queue's segment counts, and their sum.
// Two counters a thread of kThinBlock (one of kThinFusedBlock).  Every thread must call it.
__device__ __forceinline__ unsigned thin_prefix(const ThinArgs& a, unsigned L, unsigned* pre, unsigned* tmp) {
    const uint32_t* row = a.count + (L % 3) * kThinMaxSegs;
    const unsigned per = kThinMaxSegs / blockDim.x, t = threadIdx.x;
    unsigned x[2] = {row[t * per], per > 1 ? row[t * per + 1] : 0u};
    unsigned total;
    const unsigned ex = block_exclusive_scan(x[0] + x[1], tmp, total);
    pre[t * per] = ex + x[0];
    if (per > 1) pre[t * per + 1] = ex + x[0] + x[1];
    __syncthreads();
    return total;
}

__device__ __forceinline__ uint32_t thin_entry(const ThinArgs& a, const uint32_t* queue, const unsigned* pre,
                                               unsigned e) {
    const uint32_t s = find_segment(pre, a.segs, e);
    return queue[(size_t(s) << (6 + a.shift)) + (e - (s ? pre[s - 1] : 0u))];
}

__device__ __forceinline__ void thin_append(const ThinArgs& a, uint32_t* queue, uint32_t* counts, uint32_t u) {
    const uint32_t s = u >> (6 + a.shift);
    queue[(size_t(s) << (6 + a.shift)) + atomicAdd(counts + s, 1u)] = u;
}

// List entries a thread takes at once: a whole list on a grid with shortcuts, so that one
// longer list does not put a second chain of round trips on its wave.  Entries past the
// list's end are read (the list array is padded by a step) and not used.
constexpr int kThinStep = 8;
static_assert(kThinStep <= kBatchTd, "the pad of the list array");
__device__ __forceinline__ void thin_neighbours(const GraphView& g, uint32_t p, uint32_t (&u)[kThinStep]) {
#pragma unroll
    for (int j = 0; j < kThinStep; j += 4) {
        const u32x4_a4 four = *reinterpret_cast<const u32x4_a4*>(g.csrIdx + p + j);
#pragma unroll
        for (int i = 0; i < 4; ++i) u[j + i] = four[i];
    }
}

// The traversal has ended with `levels` levels (one workgroup; edges complete).
__device__ __forceinline__ void thin_finish(const ThinArgs& a, unsigned levels, unsigned shift, unsigned visited,
                                            unsigned long long* tmp64) {
    unsigned long long e = 0;
    for (uint32_t i = threadIdx.x; i < kThinMaxSegs; i += blockDim.x) e += a.edges[i];
    e = block_sum_u64(e, tmp64);
    if (threadIdx.x == 0) {
        Ctrl* c = a.ctrl;
        c->levels = levels;
        c->fusedLevels = shift;
        c->tdLevels = levels;
        c->buLevels = 0;
        c->visited = visited;
        c->visitedEdges = e;
        c->buMask = 0;
        __hip_atomic_store(&c->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// A workgroup keeps its discoveries in LDS, numbered within their segment, and takes each
// segment's room with one atomic: queue order follows vertex order, so 512 consecutive
// entries discover into a few segments.  (An atomic per discovery on the 1,024 counters
// serialised on their 32 cache lines: 200 us for a level of 330 K vertices.)  It writes them
// out after its last entries, and before that whenever it holds so many that its next 512
// entries, at most kThinMaxDegree discoveries each, might not fit; only lists longer than
// that can still overflow, and are appended one by one.  (2,048 held and the rest appended
// one by one: first BFS of the 7-ary tree of 4 M vertices 1,852 us, this way 393.)
constexpr unsigned kThinHeld = 2048;
constexpr unsigned kThinFound = kThinHeld + kThinBlock * kThinMaxDegree;

__global__ void __launch_bounds__(kThinBlock) thin_level_kernel(GraphView g, ThinArgs a, unsigned Lk) {
    const unsigned L = level_of(a.ctrl, a.levelFromCtrl, Lk);
    __shared__ unsigned pre[kThinMaxSegs], tmp[16];
    __shared__ unsigned long long tmp64[16];
    __shared__ unsigned sCnt[kThinMaxSegs], room[kThinMaxSegs], sFound;
    __shared__ uint2 found[kThinFound];  // (vertex, number within the segment)
    Ctrl* c = a.ctrl;
    const unsigned done = ld_relaxed(&c->done);
    const LevelState in = c->state[(L - 1) & 1];
    for (unsigned i = threadIdx.x; i < kThinMaxSegs; i += kThinBlock) sCnt[i] = 0;
    if (threadIdx.x == 0) sFound = 0;
    const unsigned total = thin_prefix(a, L, pre, tmp);  // its barriers publish the zeros
    if (done) return;
    const unsigned Le = L + in.shift;  // the level's distance
    if (total == 0) {
        if (blockIdx.x == 0) thin_finish(a, Le - 1, in.shift, in.visited, tmp64);
        return;
    }
    const unsigned tid = blockIdx.x * kThinBlock + threadIdx.x, nthreads = gridDim.x * kThinBlock;
    for (uint32_t i = tid; i < kThinMaxSegs; i += nthreads) a.count[((L + 2) % 3) * kThinMaxSegs + i] = 0u;
    if (tid == 0) {
        c->state[L & 1] = LevelState{0, total, in.visited + total, 0, 0, in.shift, 0ull, 0ull};
        // where the next traversal's one-workgroup kernel should take over
        c->tailFrom = total < in.prevNf && total <= kThinCap ? (c->tailFrom ? c->tailFrom : L) : 0u;
    }
    if (blockIdx.x * kThinBlock >= total) return;  // nothing for this workgroup
    const uint32_t* qin = (L & 1) ? a.queue1 : a.queue0;
    uint32_t* qout = (L & 1) ? a.queue0 : a.queue1;
    uint32_t* counts = a.count + ((L + 1) % 3) * kThinMaxSegs;
    // every thread, the list complete: room in each segment, then the entries
    const auto write_out = [&] {
        for (unsigned i = threadIdx.x; i < kThinMaxSegs; i += kThinBlock)
            if (sCnt[i]) room[i] = atomicAdd(counts + i, sCnt[i]);
        __syncthreads();
        const unsigned nf = min(sFound, kThinFound);
        for (unsigned k = threadIdx.x; k < nf; k += kThinBlock) {
            const uint32_t s = found[k].x >> (6 + a.shift);
            qout[(size_t(s) << (6 + a.shift)) + room[s] + found[k].y] = found[k].x;
        }
    };
    unsigned edges = 0;
    for (unsigned e0 = blockIdx.x * kThinBlock; e0 < total; e0 += nthreads) {  // the same for the workgroup
        const unsigned e = e0 + threadIdx.x;
        const uint32_t v = e < total ? thin_entry(a, qin, pre, e) : 0u;
        const u32x2_a4 d = *reinterpret_cast<const u32x2_a4*>(g.csrPtr + v);
        const uint32_t end = e < total ? d.y : d.x;
        edges += end - d.x;
        for (uint32_t p = d.x; p < end; p += kThinStep) {
            uint32_t u[kThinStep], w[kThinStep];
            thin_neighbours(g, p, u);
#pragma unroll
            for (int j = 0; j < kThinStep; ++j) w[j] = p + j < end ? a.visited[u[j] >> 5] : ~0u;
            // not yet visited (a stale word only shows fewer bits: the atomic decides)
#pragma unroll
            for (int j = 0; j < kThinStep; ++j) {
                const uint32_t bit = 1u << (u[j] & 31);
                w[j] = (w[j] & bit) ? ~0u : atomicOr(&a.visited[u[j] >> 5], bit);
            }
#pragma unroll
            for (int j = 0; j < kThinStep; ++j)
                if (!((w[j] >> (u[j] & 31)) & 1u)) {
                    a.levels[u[j]] = int32_t(Le);
                    const unsigned k = atomicAdd(&sFound, 1u);
                    if (k < kThinFound) found[k] = make_uint2(u[j], atomicAdd(&sCnt[u[j] >> (6 + a.shift)], 1u));
                    else thin_append(a, qout, counts, u[j]);
                }
        }
        if (e0 + nthreads >= total) break;
        __syncthreads();
        const bool full = sFound > kThinHeld;
        __syncthreads();  // every thread has read
        if (!full) continue;
        write_out();
        __syncthreads();
        for (unsigned i = threadIdx.x; i < kThinMaxSegs; i += kThinBlock) sCnt[i] = 0;
        if (threadIdx.x == 0) sFound = 0;
        __syncthreads();
    }
    const unsigned long long sum = block_sum_u64(edges, tmp64);  // its barriers complete the list
    if (threadIdx.x == 0 && sum) a.edges[blockIdx.x] += sum;     // this workgroup's alone
    write_out();
}

// Small levels back to back in one workgroup, the queue in LDS: enqueued after the init
// kernel and after each chunk of level kernels, like bfs_fused_kernel, and handing back the
// same way (the inputs of enqueued level Lk, with the levels run here in its state's shift).
__global__ void __launch_bounds__(kThinFusedBlock) thin_fused_kernel(GraphView g, ThinArgs a, unsigned Lk) {
    const unsigned L = level_of(a.ctrl, a.levelFromCtrl, Lk);
    __shared__ unsigned pre[kThinMaxSegs], tmp[16];
    __shared__ unsigned long long tmp64[16];
    __shared__ uint32_t queue[2][kThinCap];
    __shared__ unsigned sCount[2];
    Ctrl* c = a.ctrl;
    const unsigned t = threadIdx.x;
    const unsigned done = ld_relaxed(&c->done);
    const LevelState in = c->state[(L - 1) & 1];
    const unsigned total = thin_prefix(a, L, pre, tmp);
    if (done) return;
    if (total > (total < in.prevNf ? kThinCap : kThinEnter)) return;
    uint32_t* glb = (L & 1) ? a.queue1 : a.queue0;
    uint32_t* counts = a.count + (L % 3) * kThinMaxSegs;
    for (unsigned e = t; e < total; e += kThinFusedBlock) queue[0][e] = thin_entry(a, glb, pre, e);
    if (t == 0 && total && !c->tailFrom) c->tailFrom = L;
    __syncthreads();
    // the queue is in LDS: its place takes the frontier handed back
    for (uint32_t i = t; i < kThinMaxSegs; i += kThinFusedBlock) counts[i] = 0u;
    if (t < 2) sCount[t] = 0;
    __syncthreads();
    unsigned Lcur = L + in.shift, nq = total, prevNq = in.prevNf, visited = in.visited;
    unsigned long long edges = 0;
    for (unsigned it = 0;; ++it) {
        const uint32_t* q = queue[it & 1];
        uint32_t* qn = queue[(it + 1) & 1];
        unsigned* appended = &sCount[it & 1];
        if (nq == 0 || (it > 0 && nq > (nq < prevNq ? kThinCap : kThinEnter))) {
            edges = block_sum_u64(edges, tmp64);
            if (t == 0) a.edges[0] += edges;
            if (nq == 0) {
                __syncthreads();  // edges[0] is read below by another thread
                thin_finish(a, Lcur - 1, Lcur - L, visited, tmp64);
                return;
            }
            for (unsigned i = t; i < min(nq, kThinCap); i += kThinFusedBlock) thin_append(a, glb, counts, q[i]);
            if (t == 0) c->state[(L - 1) & 1] = LevelState{0, prevNq, visited, 0, 0, Lcur - L, 0ull, 0ull};
            return;
        }
        for (unsigned i = t; i < nq; i += kThinFusedBlock) {
            const u32x2_a4 d = *reinterpret_cast<const u32x2_a4*>(g.csrPtr + q[i]);
            edges += d.y - d.x;
            for (uint32_t p = d.x; p < d.y; p += kThinStep) {
                uint32_t u[kThinStep], w[kThinStep];
                thin_neighbours(g, p, u);
#pragma unroll
                for (int j = 0; j < kThinStep; ++j)
                    w[j] = p + j < d.y ? atomicOr(&a.visited[u[j] >> 5], 1u << (u[j] & 31)) : ~0u;
#pragma unroll
                for (int j = 0; j < kThinStep; ++j)
                    if (!((w[j] >> (u[j] & 31)) & 1u)) {
                        a.levels[u[j]] = int32_t(Lcur);
                        const unsigned pos = atomicAdd(appended, 1u);
                        if (pos < kThinCap) qn[pos] = u[j];
                        else thin_append(a, glb, counts, u[j]);  // the next level is handed back
                    }
            }
        }
        __syncthreads();
        visited += nq;
        prevNq = nq;
        nq = *appended;
        ++Lcur;
        if (t == 0) sCount[(it + 1) & 1] = 0;
        __syncthreads();
    }
}

}  // namespace dev
}  // namespace blest
