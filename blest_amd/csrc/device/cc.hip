// Connected components over the HBM-resident BVSS (gfx950).
//
// Reference: BVSSCCKernel (CC/BVSSCCKernel.cuh:33-276 min-label propagation over the
// BVSS, 1067-1311 host side).  The reference's fixed point is, for an undirected
// graph, the smallest (reordered) vertex ID of each component; its host compaction
// (CC/BVSSCCKernel.cuh:1269-1290) is not reproduced, labels are canonicalised to the
// smallest ORIGINAL vertex ID of the component instead.
//
// algo 0 (default): hook + compress, roots linked larger-under-smaller with a
//   compare-and-swap, independent of diameter.  With the CSR resident: a seed forest, a
//   few sampled neighbours, then only the vertices outside the largest tree.  Without it:
//   every slice (row i, mask m) of rset r is the set of edges {i, 8r+b : bit b of m},
//   each undirected edge hooked once (i < 8r+b).
// algo 1: min-label propagation, the reference's iteration (frontier = rsets whose
//   labels dropped), two stream-ordered kernels per iteration.
#include "dgraph.hpp"

namespace blest {
namespace dev {

__device__ __forceinline__ uint32_t ld_parent(const uint32_t* p, uint32_t x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Root of x with path halving.  A parent always names an ancestor, so concurrent halving
// stores keep the forest valid.
__device__ __forceinline__ uint32_t find_root(uint32_t* p, uint32_t x) {
    uint32_t par = ld_parent(p, x);
    while (par != x) {
        const uint32_t gp = ld_parent(p, par);
        if (gp == par) return par;
        __hip_atomic_store(p + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = gp;
        par = ld_parent(p, x);
    }
    return x;
}

__device__ __forceinline__ void hook(uint32_t* p, uint32_t a, uint32_t b) {
    for (;;) {
        uint32_t ra = find_root(p, a), rb = find_root(p, b);
        if (ra == rb) return;
        if (ra > rb) {
            const uint32_t t = ra;
            ra = rb;
            rb = t;
        }
        uint32_t expected = rb;
        if (__hip_atomic_compare_exchange_strong(p + rb, &expected, ra, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
        a = ra;
        b = expected;  // rb was hooked meanwhile: continue from its new parent
    }
}

__global__ void cc_init_kernel(uint32_t* p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = i;
}

__device__ __forceinline__ void hook_slice(uint32_t* p, uint32_t row, uint32_t m, uint32_t colBase) {
    for (; m; m &= m - 1) {
        const uint32_t col = colBase + __builtin_ctz(m);
        if (row < col) hook(p, row, col);
    }
}

// Wave per 64 vsets, load-balanced over their quads (as the BFS expansion).
__global__ void __launch_bounds__(256) cc_hook_kernel(GraphView g, uint32_t* p) {
    const unsigned lane = lane_id();
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned wave = tid / kWave, nwaves = (gridDim.x * blockDim.x) / kWave;
    for (unsigned base = wave * kWave; base < g.V; base += nwaves * kWave) {
        const unsigned v = base + lane;
        uint32_t q0 = 0, qc = 0, r = 0;
        if (v < g.V) {
            q0 = g.unitQuad[v];
            qc = g.unitQuad[v + 1] - q0;
            r = g.unitRset[v];
        }
        const unsigned incl = wave_inclusive_scan(qc);
        const unsigned excl = incl - qc;
        const unsigned total = __shfl(incl, kWave - 1, kWave);
        for (unsigned t0 = 0; t0 < total; t0 += kWave) {
            const unsigned t = t0 + lane;
            const unsigned owner = wave_owner(excl, min(t, total - 1));
            const uint32_t oq0 = __shfl(q0, owner, kWave);
            const unsigned oex = __shfl(excl, owner, kWave);
            const uint32_t orr = __shfl(r, owner, kWave);
            if (t < total) {
                const uint32_t q = oq0 + (t - oex);
                const uint4 r4 = g.rows[q];
                const uint32_t m = g.masks[q];
                const uint32_t cb = orr * 8;
                hook_slice(p, r4.x, m & 0xFF, cb);
                hook_slice(p, r4.y, (m >> 8) & 0xFF, cb);
                hook_slice(p, r4.z, (m >> 16) & 0xFF, cb);
                hook_slice(p, r4.w, (m >> 24) & 0xFF, cb);
            }
        }
    }
}

// Parents read through the CU's own cache: an old value is an old ancestor (a parent only
// ever moves up its own tree), and a root that looks like one but no longer is loses its
// compare-and-swap and goes on from the value that returns.
__device__ __forceinline__ uint32_t ld_parent_near(const uint32_t* p, uint32_t x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// After hooking the roots are final.  Compression must store roots only: a
// path-halving store (an ancestor that is not the root) racing with another thread's
// final store could overwrite it.  Every value a thread can read here (an old parent or
// a root) is an ancestor, so the read-only walk always ends at the root.
__global__ void cc_compress_kernel(uint32_t* p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        uint32_t x = i, par = ld_parent_near(p, x);
        while (par != x) {
            x = par;
            par = ld_parent_near(p, x);
        }
        if (x != i) __hip_atomic_store(p + i, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ----------------------------------------------- components from the CSR (algo 0)
// Hooking every edge of the graph costs a pass over all slices with two dependent walks
// per edge, and on a social graph the concurrent compare-and-swaps meet at the hubs'
// roots.  With the (symmetric) CSR resident almost no edge needs to be hooked.  The plan (hook
// sampled neighbours, compress, find the most frequent tree, finish only what lies outside
// it) is that of Afforest (Sutton, Ben-Nun and Barak, "Optimizing Parallel Graph Connectivity
// Computation via Subgraph Sampling", IPDPS 2018); the seed forest, the hooks and the minima
// are this kernel's own:
//   seed    a vertex takes its highest-degree neighbour (the first of its list) as
//           parent when that neighbour ranks above it: (degree, smaller ID).  Ranks rise
//           along parents, so this is a forest, made without one atomic;
//   sample  each vertex hooks its first neighbour, then (the trees compressed) its next
//           kCcSampled ones; after that nearly every vertex of a large component hangs
//           under one root;
//   giant   the most frequent root among kCcVotes sampled vertices;
//   rest    only vertices outside that tree hook the rest of their lists (an edge that
//           leaves the tree is in the list of its outer end too: the graph is symmetric).
// Hooks link roots only, larger ID under smaller, so a root is hooked at most once and
// the links between roots fall in ID: no cycle whatever the seed forest's order was.
// Roots are no longer the smallest vertices of their components; the labels come from
// the minimum taken over each tree at the end.
// Bound by the launches and the dependent walks, not by memory (R-MAT 20: 8 MB of
// offsets, probes and parents).  Measured (MI355X, whole call): R-MAT 20 natural order,
// labels on the device, 1.5-3.9 ms with every slice hooked (by the graph's seed) ->
// 0.142 ms; 1023-square grid in RCM order, labels to the host, 13.2 -> 0.48 ms.
constexpr uint32_t kCcSampled = 2;
constexpr unsigned kCcVotes = 256;
constexpr uint32_t kCcHeavy = 64;  // longer lists are hooked by a whole wave
constexpr int kCcBlock = 256;

// Reads only: a halving store of values that lag behind could put an older, lower ancestor
// back in the place of a newer one.
__device__ __forceinline__ uint32_t find_root_near(const uint32_t* p, uint32_t x) {
    uint32_t par = ld_parent_near(p, x);
    while (par != x) {
        x = par;
        par = ld_parent_near(p, x);
    }
    return x;
}

__device__ __forceinline__ void hook_near(uint32_t* p, uint32_t a, uint32_t b) {
    uint32_t ra = find_root_near(p, a), rb = find_root_near(p, b);
    if (ra == rb) return;
    for (;;) {
        // the CU's own copy may lag behind: go on to the current roots before the swap (a
        // swap that fails meets every other one at that root, a load does not)
        ra = find_root(p, ra);
        rb = find_root(p, rb);
        if (ra == rb) return;
        if (ra > rb) {
            const uint32_t t = ra;
            ra = rb;
            rb = t;
        }
        uint32_t expected = rb;
        if (__hip_atomic_compare_exchange_strong(p + rb, &expected, ra, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
        rb = expected;  // rb was hooked meanwhile: go on from its parent
    }
}

// p = the seed forest, minOf = no minimum yet.  A workgroup takes kCcTile consecutive vertices,
// one a thread, and follows their parents inside the tile in LDS (pointer doubling) before it
// writes them: among equal degrees parents fall in ID, so on a graph numbered along its
// paths (a road, a band matrix) a tree is a chain over all of them, and the compression after
// this walks it link by link from every vertex.  A chain's vertices within a tile follow each
// other, so it leaves here with a link per tile and degree.  (Whole call, without and with:
// path of 1 M vertices 1864 and 142 us, of 200 K 661 and 102; R-MAT 20, whose first
// neighbours lie in other tiles, 145 and 143.)
constexpr int kCcTile = 1024;

__global__ void __launch_bounds__(kCcTile) cc_seed_kernel(GraphView g, uint32_t* p, uint32_t* minOf) {
    __shared__ uint32_t up[kCcTile], parent[kCcTile];
    const uint32_t t = threadIdx.x;
    for (uint64_t v0 = uint64_t(blockIdx.x) * kCcTile; v0 < g.n; v0 += uint64_t(gridDim.x) * kCcTile) {
        const bool ok = v0 + t < g.n;
        const uint32_t v = uint32_t(v0) + t;
        uint32_t par = v;
        if (ok) {
            const uint32_t b = g.csrPtr[v], deg = g.csrPtr[v + 1] - b;
            if (deg) {
                const uint32_t u = g.probe ? g.probe[v] : g.csrIdx[b];
                const uint32_t du = g.csrPtr[u + 1] - g.csrPtr[u];
                if (du > deg || (du == deg && u < v)) par = u;
            }
            minOf[v] = 0xFFFFFFFFu;
        }
        const uint32_t local = par - uint32_t(v0);
        uint32_t x = local < uint32_t(kCcTile) ? local : t;  // last vertex reached inside the tile
        parent[t] = par;
        up[t] = x;
        __syncthreads();
        while (__syncthreads_or(up[x] != x)) {
            const uint32_t y = up[x];
            __syncthreads();  // every thread has read
            up[t] = x = y;
            __syncthreads();
        }
        if (ok) p[v] = parent[x];
        __syncthreads();  // the next tile reuses the arrays
    }
}

// Hooks entries [first, last) of every vertex's list; trees already joined are told apart
// by one load each (p is compressed).
__global__ void __launch_bounds__(kCcBlock) cc_sample_hook_kernel(GraphView g, uint32_t* p, uint32_t first,
                                                                  uint32_t last) {
    for (uint32_t v = blockIdx.x * kCcBlock + threadIdx.x; v < g.n; v += gridDim.x * kCcBlock) {
        const uint32_t b = g.csrPtr[v], e = g.csrPtr[v + 1];
        for (uint32_t i = part_end(b, e, first); i < part_end(b, e, last); ++i) {
            const uint32_t u = g.csrIdx[i];
            if (ld_parent_near(p, u) != ld_parent_near(p, v)) hook_near(p, v, u);
        }
    }
}

// giant[0] = the root that most of the sampled vertices hang under (one workgroup; p is
// compressed).  Each thread counts the votes for its own sample's root.  The rest's hooks may
// link that root under another: cc_min_original_kernel leaves the tree's final root in giant[1].
__global__ void __launch_bounds__(kCcVotes) cc_giant_kernel(const uint32_t* p, uint32_t n, uint32_t* giant) {
    __shared__ uint32_t root[kCcVotes];
    __shared__ unsigned long long best;
    const unsigned t = threadIdx.x;
    const uint32_t r = p[uint64_t(t) * n / kCcVotes];
    root[t] = r;
    if (t == 0) best = 0;
    __syncthreads();
    unsigned votes = 0;
    for (unsigned i = 0; i < kCcVotes; ++i) votes += root[i] == r;
    atomicMax(&best, (unsigned long long)votes << 32 | r);
    __syncthreads();
    if (t == 0) giant[0] = uint32_t(best);
}

__global__ void __launch_bounds__(kCcBlock) cc_rest_kernel(GraphView g, uint32_t* p, const uint32_t* giant) {
    const unsigned lane = lane_id();
    const uint32_t big = giant[0];
    const uint32_t n64 = (g.n + kWave - 1) / kWave * kWave;  // whole waves: the ballots below
    for (uint32_t v = blockIdx.x * kCcBlock + threadIdx.x; v < n64; v += gridDim.x * kCcBlock) {
        uint32_t b = 0, e = 0;
        if (v < g.n && ld_parent_near(p, v) != big) {
            e = g.csrPtr[v + 1];
            b = part_end(g.csrPtr[v], e, kCcSampled + 1);
        }
        const bool heavy = b < e && e - b > kCcHeavy;
        if (!heavy)
            for (uint32_t i = b; i < e; ++i) hook_near(p, v, g.csrIdx[i]);
        for (unsigned long long h = __ballot(heavy); h; h &= h - 1) {
            const int l = __builtin_ctzll(h);
            const uint32_t hv = __shfl(v, l, kWave), hb = __shfl(b, l, kWave), he = __shfl(e, l, kWave);
            for (uint32_t i = lane; in_part(hb, i, he); i += kWave) hook_near(p, hv, g.csrIdx[hb + i]);
        }
    }
}

// minOf[root] = smallest original ID in the component (the giant tree's as one minimum per
// workgroup, giantMin), and the number of roots per workgroup (their sum is the component
// count).  A wave carries the running minimum of the root it met last in a register and
// gives it up, one atomic, when another root takes its place or at the end; an atomic is
// only issued when it would lower the value.  (An atomicMin per vertex serialised at the
// giant component's address: 11.9 ms for the 1 M vertices of a 1023-square grid; one per
// wave still 71 us there and 230 us on R-MAT 20.)
__device__ __forceinline__ void lower_min(uint32_t* minOf, uint32_t root, uint32_t id) {
    if (id < __hip_atomic_load(minOf + root, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(minOf + root, id);
}

__global__ void __launch_bounds__(kCcBlock) cc_min_original_kernel(const uint32_t* p, const uint32_t* newToOld,
                                                                   uint32_t* minOf, uint32_t* giant,
                                                                   uint32_t* giantMin, uint32_t* rootsPerBlock,
                                                                   uint32_t n) {
    __shared__ unsigned long long tmp64[16];
    __shared__ uint32_t blockMin;
    const unsigned lane = lane_id();
    const uint32_t big = p[giant[0]];
    if (threadIdx.x == 0) blockMin = 0xFFFFFFFFu;
    __syncthreads();
    uint32_t bigMin = 0xFFFFFFFFu;
    uint32_t held = 0xFFFFFFFFu, heldMin = 0xFFFFFFFFu, roots = 0;  // held: wave-uniform
    const uint32_t n64 = (n + kWave - 1) / kWave * kWave;
    for (uint32_t i = blockIdx.x * kCcBlock + threadIdx.x; i < n64; i += gridDim.x * kCcBlock) {
        const bool ok = i < n;
        const uint32_t r = ok ? p[i] : 0xFFFFFFFFu;
        const uint32_t id = ok ? (newToOld ? newToOld[i] : i) : 0xFFFFFFFFu;
        roots += r == i;
        bool left = ok && r != big;
        if (ok && !left) bigMin = min(bigMin, id);
        // the root met last, then the roots of the first two lanes that differ; the rest
        // are small components, whose lanes go alone
        for (int round = 0; round < 3; ++round) {
            const unsigned long long open = __ballot(left);
            if (!open) break;
            const uint32_t cand = round == 0 ? held : uint32_t(__shfl(r, __builtin_ctzll(open), kWave));
            const unsigned long long same = __ballot(left && r == cand);
            if (!same) continue;
            if (__popcll(same) == 1 && cand != held) {  // alone: no reduction, nothing replaced
                if (left && r == cand) lower_min(minOf, r, id);
            } else {
                uint32_t m = left && r == cand ? id : 0xFFFFFFFFu;
                for (int d = kWave / 2; d > 0; d >>= 1) m = min(m, uint32_t(__shfl_xor(m, d, kWave)));
                if (cand != held) {
                    if (lane == 0 && held != 0xFFFFFFFFu) lower_min(minOf, held, heldMin);
                    held = cand;
                    heldMin = m;
                } else {
                    heldMin = min(heldMin, m);
                }
            }
            left = left && r != cand;
        }
        if (left) lower_min(minOf, r, id);
    }
    if (lane == 0 && held != 0xFFFFFFFFu) lower_min(minOf, held, heldMin);
    atomicMin(&blockMin, bigMin);  // LDS
    const unsigned long long total = block_sum_u64(roots, tmp64);  // its barriers complete blockMin
    if (threadIdx.x == 0) {
        rootsPerBlock[blockIdx.x] = uint32_t(total);
        giantMin[blockIdx.x] = blockMin;
        if (blockIdx.x == 0) giant[1] = big;
    }
}

__global__ void fill_u32_kernel(uint32_t* a, uint32_t v, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

// out[old] = minOf[root(new(old))]; launched with the grid of cc_min_original_kernel, whose
// workgroups left one minimum of the giant tree each.
__global__ void __launch_bounds__(kCcBlock) cc_relabel_kernel(const uint32_t* p, const uint32_t* oldToNew,
                                                              const uint32_t* minOf, const uint32_t* giant,
                                                              const uint32_t* giantMin, uint32_t* out, uint32_t n) {
    __shared__ uint32_t all;
    const uint32_t big = giant[1];
    if (threadIdx.x == 0) all = 0xFFFFFFFFu;
    __syncthreads();
    uint32_t m = 0xFFFFFFFFu;
    for (uint32_t i = threadIdx.x; i < gridDim.x; i += kCcBlock) m = min(m, giantMin[i]);
    atomicMin(&all, m);  // LDS
    __syncthreads();
    const uint32_t bigMin = all;
    for (uint32_t i = blockIdx.x * kCcBlock + threadIdx.x; i < n; i += gridDim.x * kCcBlock) {
        const uint32_t r = p[oldToNew ? oldToNew[i] : i];
        out[i] = r == big ? bigMin : minOf[r];
    }
}

// ------------------------------------------------------------ label propagation
struct LpArgs {
    uint32_t* labels;
    unsigned long long* front0;
    unsigned long long* front1;
    unsigned long long* marker;
    uint32_t* list0;
    uint32_t* list1;
    Ctrl* ctrl;
    SegView sv;
    SegCounters sc;
};

__device__ __forceinline__ void lp_slice(uint32_t* labels, unsigned long long* marker, uint32_t row, uint32_t valid,
                                         uint32_t colBase) {
    if (!valid) return;
    uint32_t best = ld_parent(labels, row);
    const uint32_t mine = best;
    for (; valid; valid &= valid - 1) best = min(best, ld_parent(labels, colBase + __builtin_ctz(valid)));
    if (best < mine) {
        const uint32_t old = atomicMin(labels + row, best);
        if (best < old) atomicOr(&marker[row >> 6], 1ull << (row & 63));
    }
}

// All vertices start active; every vset is in the first list (CC/BVSSCCKernel.cuh:1084-1088,
// 1183-1203).
__global__ void __launch_bounds__(kProducerBlock) cc_lp_init_kernel(GraphView g, LpArgs a) {
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x, nthreads = gridDim.x * blockDim.x;
    for (uint32_t i = tid; i < g.n; i += nthreads) a.labels[i] = i;
    for (uint32_t w = tid; w < g.W; w += nthreads) {
        const uint32_t cnt = min(64u, g.n - w * 64);
        a.front1[w] = cnt == 64 ? ~0ull : ((1ull << cnt) - 1);
        a.marker[w] = 0ull;
    }
    // every segment lists all of its vsets
    for (uint32_t v = tid; v < g.V; v += nthreads) a.list1[v] = v;
    for (uint32_t s = tid; s < a.sv.segs; s += nthreads)
        a.sc.count[a.sv.segs + s] = a.sv.segBase[s + 1] - a.sv.segBase[s];
    if (tid == 0) a.ctrl->done = 0;
}

// Iteration L: every slice of a listed vset whose mask meets its rset's active byte
// lowers its row's label to the smallest active column label (CC/BVSSCCKernel.cuh:67-221).
__global__ void __launch_bounds__(kProducerBlock) cc_lp_expand_kernel(GraphView g, LpArgs a, unsigned L) {
    __shared__ unsigned pre[kMaxSegs];
    __shared__ unsigned tmp[16];
    Ctrl* c = a.ctrl;
    if (ld_relaxed(&c->done)) return;
    const unsigned cnt = load_prefix(a.sc.count + size_t(L % 3) * a.sv.segs, a.sv.segs, pre, tmp);
    if (cnt == 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            c->iterations = L - 1;
            __hip_atomic_store(&c->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    const unsigned lane = lane_id();
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned wave = tid / kWave, nwaves = (gridDim.x * blockDim.x) / kWave;
    const unsigned long long* fin = (L & 1) ? a.front1 : a.front0;
    const uint32_t* lin = (L & 1) ? a.list1 : a.list0;
    for (unsigned base = wave * kWave; base < cnt; base += nwaves * kWave) {
        const unsigned e = base + lane;
        uint32_t q0 = 0, qc = 0, fb = 0, r = 0;
        if (e < cnt) {
            const uint32_t v = list_entry(lin, a.sv, pre, e);
            q0 = g.unitQuad[v];
            qc = g.unitQuad[v + 1] - q0;
            r = g.unitRset[v];
            fb = reinterpret_cast<const uint8_t*>(fin)[r];
            if (!fb) qc = 0;
        }
        const unsigned incl = wave_inclusive_scan(qc);
        const unsigned excl = incl - qc;
        const unsigned total = __shfl(incl, kWave - 1, kWave);
        for (unsigned t0 = 0; t0 < total; t0 += kWave) {
            const unsigned t = t0 + lane;
            const unsigned owner = wave_owner(excl, min(t, total - 1));
            const uint32_t oq0 = __shfl(q0, owner, kWave);
            const unsigned oex = __shfl(excl, owner, kWave);
            const uint32_t of = __shfl(fb, owner, kWave);
            const uint32_t orr = __shfl(r, owner, kWave);
            if (t < total) {
                const uint32_t q = oq0 + (t - oex);
                const uint4 r4 = g.rows[q];
                const uint32_t m = g.masks[q];
                const uint32_t cb = orr * 8;
                lp_slice(a.labels, a.marker, r4.x, m & of & 0xFF, cb);
                lp_slice(a.labels, a.marker, r4.y, (m >> 8) & of & 0xFF, cb);
                lp_slice(a.labels, a.marker, r4.z, (m >> 16) & of & 0xFF, cb);
                lp_slice(a.labels, a.marker, r4.w, (m >> 24) & of & 0xFF, cb);
            }
        }
    }
}

// Marked vertices become the next active set; their rsets' vsets the next list
// (CC/BVSSCCKernel.cuh:228-269).
__global__ void __launch_bounds__(kProducerBlock) cc_lp_update_kernel(GraphView g, LpArgs a, unsigned L) {
    __shared__ unsigned tmp[16];
    Ctrl* c = a.ctrl;
    if (ld_relaxed(&c->done)) return;
    unsigned long long* fout = (L & 1) ? a.front0 : a.front1;
    uint32_t* lout = (L & 1) ? a.list0 : a.list1;
    const uint32_t ws = blockIdx.x * a.sv.wps, we = min(g.W, ws + a.sv.wps);
    uint32_t* out = lout + a.sv.segBase[blockIdx.x];
    unsigned running = 0;
    for (uint32_t r0 = ws; r0 < we; r0 += blockDim.x) {
        const uint32_t w = r0 + threadIdx.x;
        unsigned long long mk = 0;
        if (w < we) {
            mk = a.marker[w];
            if (mk) a.marker[w] = 0ull;
            fout[w] = mk;
        }
        const unsigned cnt = word_vsets(g.rsetUnit, w, mk);
        unsigned tot;
        const unsigned ex = block_exclusive_scan(cnt, tmp, tot);
        // each wave writes its 64 words' vsets, balanced over its lanes
        const unsigned waveStart = __shfl(ex, 0, kWave);
        const uint32_t w0 = r0 + (threadIdx.x / kWave) * kWave;
        const uint32_t w1 = min(we, w0 + kWave);
        if (w0 < w1)
            wave_write_vsets(g.rsetUnit, w0, w1, [&](uint32_t x) { return __shfl(mk, x - w0, kWave); },
                             out + running + waveStart);
        running += tot;
    }
    if (threadIdx.x == 0) a.sc.count[size_t((L + 1) % 3) * a.sv.segs + blockIdx.x] = running;
}

}  // namespace dev

// ------------------------------------------------------------------------ host
static void cc_run(Query& q, int algo, uint32_t* hostLabels, blest_cc_stats* st) {
    DeviceGraph& g = *q.g;
    if (!g.symmetric) throw Error(BLEST_ERR_UNSUPPORTED, "connected components need a symmetric graph");
    const bool labelsOnDevice = hostLabels && check_result_range(hostLabels, 4 * size_t(g.n), g.device, "labels");
    if (algo != 0 && algo != 1) throw Error(BLEST_ERR_INVALID_ARGUMENT, "unknown CC algorithm");
    const dim3 block(dev::kCcBlock);
    const dim3 grid(std::min<uint32_t>(uint32_t(g.cus) * 8, (g.n + dev::kCcBlock - 1) / dev::kCcBlock));
    // the sampled hooks meet at the trees that swallow the rest: fewer waves at once fail
    // fewer swaps (whole call with all and a quarter of the workgroups: 300-square grid 306
    // and 190 us, mean degree 5 and 100 K vertices 441 and 204; an eighth is slower on
    // grids, 223 and 274 on the 1023-square one in RCM order)
    const dim3 few(std::max<uint32_t>(1, grid.x / 4));
    if (!q.labels) {
        // one allocation: all of it or none, so that a call that found no room leaves
        // nothing half made for the next one
        const size_t n = (size_t(g.n) + 63) / 64 * 64, counts = 2 * size_t(g.cus) * 8 + 2;
        q.hostCcCounts.resize(size_t(g.cus) * 8);
        q.labels = q.alloc<uint32_t>(2 * n + counts);
        q.labelsAux = q.labels + n;
        q.ccCounts = q.labelsAux + n;
    }
    GraphView gv = g.view();
    unsigned iterations = 1;
    uint32_t *giantMin = q.ccCounts + size_t(g.cus) * 8, *giant = giantMin + size_t(g.cus) * 8;
    const auto vote = [&] {
        hipLaunchKernelGGL(dev::cc_giant_kernel, dim3(1), dim3(dev::kCcVotes), 0, q.stream, q.labels, g.n, giant);
    };
    BLEST_HIP(hipEventRecord(q.ev0, q.stream));
    if (algo == 0 && g.hasCsr) {
        const dim3 tiles(std::min<uint32_t>(uint32_t(g.cus) * 2, (g.n - 1) / dev::kCcTile + 1));
        hipLaunchKernelGGL(dev::cc_seed_kernel, tiles, dim3(dev::kCcTile), 0, q.stream, gv, q.labels, q.labelsAux);
        hipLaunchKernelGGL(dev::cc_compress_kernel, grid, block, 0, q.stream, q.labels, g.n);
        hipLaunchKernelGGL(dev::cc_sample_hook_kernel, grid, block, 0, q.stream, gv, q.labels, 0u, 1u);
        hipLaunchKernelGGL(dev::cc_compress_kernel, grid, block, 0, q.stream, q.labels, g.n);
        hipLaunchKernelGGL(dev::cc_sample_hook_kernel, few, block, 0, q.stream, gv, q.labels, 1u,
                           dev::kCcSampled + 1u);
        hipLaunchKernelGGL(dev::cc_compress_kernel, grid, block, 0, q.stream, q.labels, g.n);
        vote();
        hipLaunchKernelGGL(dev::cc_rest_kernel, grid, block, 0, q.stream, gv, q.labels, giant);
        hipLaunchKernelGGL(dev::cc_compress_kernel, grid, block, 0, q.stream, q.labels, g.n);
        BLEST_HIP(hipGetLastError());
    } else if (algo == 0) {
        // no CSR resident: every slice's edges are hooked
        hipLaunchKernelGGL(dev::cc_init_kernel, grid, block, 0, q.stream, q.labels, g.n);
        hipLaunchKernelGGL(dev::cc_hook_kernel, dim3(uint32_t(g.cus) * 8), block, 0, q.stream, gv, q.labels);
        hipLaunchKernelGGL(dev::cc_compress_kernel, grid, block, 0, q.stream, q.labels, g.n);
        hipLaunchKernelGGL(dev::fill_u32_kernel, grid, block, 0, q.stream, q.labelsAux, 0xFFFFFFFFu, g.n);
        vote();
        BLEST_HIP(hipGetLastError());
    } else {
        dev::LpArgs a;
        a.labels = q.labels;
        a.front0 = q.front0;
        a.front1 = q.front1;
        a.marker = q.next;
        a.list0 = q.list0;
        a.list1 = q.list1;
        a.ctrl = q.ctrl;
        a.sv = g.wide_view();
        a.sc = q.seg_counters();
        const dim3 lg = wide_grid(g), lb(dev::kProducerBlock);
        hipLaunchKernelGGL(dev::cc_lp_init_kernel, lg, lb, 0, q.stream, gv, a);
        run_levels(q, [&](unsigned L) {
            hipLaunchKernelGGL(dev::cc_lp_expand_kernel, lg, lb, 0, q.stream, gv, a, L);
            hipLaunchKernelGGL(dev::cc_lp_update_kernel, lg, lb, 0, q.stream, gv, a, L);
        });
        hipLaunchKernelGGL(dev::fill_u32_kernel, grid, block, 0, q.stream, q.labelsAux, 0xFFFFFFFFu, g.n);
        vote();
        BLEST_HIP(hipGetLastError());
        iterations = q.hostCtrl->iterations;
    }
    // canonical labels, straight into the caller's array when it is device memory (host
    // results are staged: over the parents, or in the level array when the relabelling
    // permutes), and the component count
    uint32_t* result = labelsOnDevice ? hostLabels : g.hasPerm ? reinterpret_cast<uint32_t*>(q.levels) : q.labels;
    hipLaunchKernelGGL(dev::cc_min_original_kernel, grid, block, 0, q.stream, q.labels,
                       g.hasPerm ? g.permNewToOld : nullptr, q.labelsAux, giant, giantMin, q.ccCounts, g.n);
    if (hostLabels)
        hipLaunchKernelGGL(dev::cc_relabel_kernel, grid, block, 0, q.stream, q.labels,
                           g.hasPerm ? g.permOldToNew : nullptr, q.labelsAux, giant, giantMin, result, g.n);
    BLEST_HIP(hipGetLastError());
    BLEST_HIP(hipEventRecord(q.ev1, q.stream));
    BLEST_HIP(hipMemcpyAsync(q.hostCcCounts.data(), q.ccCounts, 4 * size_t(grid.x), hipMemcpyDeviceToHost, q.stream));
    if (hostLabels && !labelsOnDevice)
        BLEST_HIP(hipMemcpyAsync(hostLabels, result, 4 * size_t(g.n), hipMemcpyDefault, q.stream));
    BLEST_HIP(hipStreamSynchronize(q.stream));
    if (st) {
        float ms = 0;
        BLEST_HIP(hipEventElapsedTime(&ms, q.ev0, q.ev1));
        uint32_t comps = 0;
        for (uint32_t i = 0; i < grid.x; ++i) comps += q.hostCcCounts[i];
        st->kernel_ms = ms;
        st->no_components = comps;
        st->iterations = iterations;
    }
}

}  // namespace blest

using namespace blest;

extern "C" blest_status blest_cc(blest_query* qh, int algo, uint32_t* labels, blest_cc_stats* st) {
    return guarded([&] {
        if (!qh) throw Error(BLEST_ERR_INVALID_ARGUMENT, "query is null");
        Query& q = qh->q;
        std::lock_guard<std::mutex> lk(q.mu);
        BLEST_HIP(hipSetDevice(q.g->device));
        cc_run(q, algo, labels, st);
    });
}
