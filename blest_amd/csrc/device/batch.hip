// Many small graphs in one launch: one workgroup of 1,024 threads traverses one graph from
// its root, with the visited / frontier / next bitmaps held in LDS (n <= 131072 per graph:
// 3 x 16 KiB), so levels are separated by workgroup barriers only and no bitmap access
// leaves the CU.  The graphs are symmetric, so one CSR serves both directions.
#include <cstring>

#include "dgraph.hpp"
#include "small_traverse.hpp"

namespace blest {
namespace dev {

struct BatchGraph {
    uint32_t n;
    uint32_t narrow;     // 1: list entries are 16-bit (n <= 65536), 0: 32-bit
    uint64_t levelOff;   // into the concatenated level array
    uint64_t csrPtrOff;  // into csrPtr (n + 1 entries per graph, graph-relative)
    uint64_t csrIdxOff;  // into csrIdx, in 16-bit units (even)
};

struct BatchArgs {
    const BatchGraph* graphs;
    const uint32_t* csrPtr;
    const uint16_t* csrIdx;
    const uint32_t* roots;
    const uint32_t* order;
    int32_t* levels;
    uint32_t maxWords;
    double alpha;
};

constexpr double kBatchBeta = 24.0;  // back to top-down when the frontier falls below n / 24

__global__ void __launch_bounds__(kBatchBlock) __attribute__((amdgpu_waves_per_eu(8))) batch_bfs_kernel(BatchArgs a) {
    extern __shared__ unsigned long long lds[];
    __shared__ unsigned sNew[3];
    __shared__ unsigned long long sEdges[3];
    const uint32_t gi = a.order[blockIdx.x];
    const BatchGraph G = a.graphs[gi];
    const uint16_t* ci = a.csrIdx + G.csrIdxOff;
    const SmallGraph sg{G.n, a.csrPtr + G.csrPtrOff};
    int32_t* levels = a.levels + G.levelOff;
    if (G.narrow)
        small_traverse(sg, a.roots[gi], ci, levels, a.alpha, kBatchBeta, lds, a.maxWords, sNew, sEdges);
    else
        small_traverse(sg, a.roots[gi], reinterpret_cast<const uint32_t*>(ci), levels, a.alpha, kBatchBeta, lds,
                       a.maxWords, sNew, sEdges);
}

}  // namespace dev

struct GraphBatch {
    int device = 0;
    uint32_t count = 0, maxWords = 0;
    uint64_t totalN = 0;
    std::vector<uint32_t> sizes;
    dev::BatchGraph* graphs = nullptr;
    uint32_t *csrPtr = nullptr, *roots = nullptr;
    uint16_t* csrIdx = nullptr;
    uint32_t* order = nullptr;  // workgroup -> graph
    int32_t* levels = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<void*> allocs;
    template <class T>
    T* upload(const std::vector<T>& v) {
        void* p = nullptr;
        BLEST_HIP(hipMalloc(&p, std::max<size_t>(1, v.size()) * sizeof(T)));
        allocs.push_back(p);
        if (!v.empty()) BLEST_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
        return static_cast<T*>(p);
    }
    ~GraphBatch() {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void* p : allocs) (void)hipFree(p);
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

}  // namespace blest

struct blest_graph_batch {
    blest::GraphBatch b;
};

using namespace blest;

extern "C" {

blest_status blest_graph_batch_create(const blest_csc* const* graphs, uint32_t count, int device,
                                      blest_graph_batch** out) {
    return guarded([&] {
        if (!graphs || !out || count == 0) throw Error(BLEST_ERR_INVALID_ARGUMENT, "empty batch");
        auto* h = new blest_graph_batch();
        GraphBatch& gb = h->b;
        try {
            gb.device = device;
            BLEST_HIP(hipSetDevice(device));
            std::vector<dev::BatchGraph> info(count);
            std::vector<int> bad(count, 0);
            for (uint32_t i = 0; i < count; ++i)
                if (!graphs[i]) throw Error(BLEST_ERR_INVALID_ARGUMENT, "null graph in batch");
            parallel_dynamic(count, hw_threads(), 1, [&](uint64_t i, unsigned) {
                const CSC& g = csc_of(graphs[i]);
                if (g.n == 0 || g.n > 131072) bad[i] = 1;
                else if (!csc_is_symmetric(g, 1)) bad[i] = 2;
            });
            for (uint32_t i = 0; i < count; ++i) {
                if (bad[i] == 1) throw Error(BLEST_ERR_UNSUPPORTED, "batched graphs need 1 <= n <= 131072");
                if (bad[i] == 2) throw Error(BLEST_ERR_UNSUPPORTED, "batched graphs must be symmetric");
            }
            uint64_t lv = 0, ncp = 0, nci = 0;
            for (uint32_t i = 0; i < count; ++i) {
                const CSC& g = csc_of(graphs[i]);
                dev::BatchGraph& G = info[i];
                G.n = g.n;
                G.levelOff = lv;
                G.csrPtrOff = ncp;
                G.csrIdxOff = nci;
                lv += g.n;
                ncp += g.colPtrs.size();
                G.narrow = g.n <= 65536;
                nci += G.narrow ? (g.rows.size() + 1) / 2 * 2 : 2 * g.rows.size();
                gb.sizes.push_back(g.n);
                gb.maxWords = std::max(gb.maxWords, (g.n + 63) / 64);
            }
            std::vector<uint32_t> cpAll(ncp);
            std::vector<uint16_t> ciAll(nci + 2 * dev::kBatchTd);  // a step may read past the last list
            parallel_dynamic(count, hw_threads(), 16, [&](uint64_t i, unsigned) {
                const CSC& g = csc_of(graphs[i]);
                const dev::BatchGraph& G = info[i];
                std::copy(g.colPtrs.begin(), g.colPtrs.end(), cpAll.begin() + G.csrPtrOff);
                uint16_t* to = ciAll.data() + G.csrIdxOff;
                if (G.narrow)
                    std::transform(g.rows.begin(), g.rows.end(), to, [](uint32_t r) { return uint16_t(r); });
                else if (!g.rows.empty())
                    std::memcpy(to, g.rows.data(), 4 * g.rows.size());
            });
            // Workgroups start roughly in index order: largest graphs first, so the
            // small ones fill in behind them (longest-processing-time order).
            std::vector<uint32_t> order(count);
            for (uint32_t i = 0; i < count; ++i) order[i] = i;
            std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return info[x].n > info[y].n; });
            gb.order = gb.upload(order);
            gb.count = count;
            gb.totalN = lv;
            gb.graphs = gb.upload(info);
            gb.csrPtr = gb.upload(cpAll);
            gb.csrIdx = gb.upload(ciAll);
            gb.roots = gb.upload(std::vector<uint32_t>(count, 0));
            gb.levels = gb.upload(std::vector<int32_t>(lv, 0));
            BLEST_HIP(hipStreamCreateWithFlags(&gb.stream, hipStreamNonBlocking));
            BLEST_HIP(hipEventCreate(&gb.ev0));
            BLEST_HIP(hipEventCreate(&gb.ev1));
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

void blest_graph_batch_free(blest_graph_batch* gb) { delete gb; }

blest_status blest_graph_batch_bfs(blest_graph_batch* h, const uint32_t* roots, int32_t* levels, double* kernel_ms) {
    return guarded([&] {
        if (!h || !roots) throw Error(BLEST_ERR_INVALID_ARGUMENT, "null argument");
        GraphBatch& gb = h->b;
        BLEST_HIP(hipSetDevice(gb.device));
        for (uint32_t i = 0; i < gb.count; ++i)
            if (roots[i] >= gb.sizes[i]) throw Error(BLEST_ERR_INVALID_ARGUMENT, "root out of range");
        // device results are written in place, host ones staged in gb.levels
        const bool onDevice = levels && check_result_range(levels, 4 * size_t(gb.totalN), gb.device, "levels");
        BLEST_HIP(hipMemcpyAsync(gb.roots, roots, 4 * size_t(gb.count), hipMemcpyHostToDevice, gb.stream));
        dev::BatchArgs a;
        a.graphs = gb.graphs;
        a.csrPtr = gb.csrPtr;
        a.csrIdx = gb.csrIdx;
        a.roots = gb.roots;
        a.order = gb.order;
        a.levels = onDevice ? levels : gb.levels;
        a.maxWords = gb.maxWords;
        a.alpha = 4.0;
        const size_t lds = size_t(3) * gb.maxWords * sizeof(unsigned long long);
        BLEST_HIP(hipEventRecord(gb.ev0, gb.stream));
        hipLaunchKernelGGL(dev::batch_bfs_kernel, dim3(gb.count), dim3(dev::kBatchBlock), lds, gb.stream, a);
        BLEST_HIP(hipGetLastError());
        BLEST_HIP(hipEventRecord(gb.ev1, gb.stream));
        if (levels && !onDevice)
            BLEST_HIP(hipMemcpyAsync(levels, gb.levels, 4 * gb.totalN, hipMemcpyDefault, gb.stream));
        BLEST_HIP(hipStreamSynchronize(gb.stream));
        float ms = 0;
        BLEST_HIP(hipEventElapsedTime(&ms, gb.ev0, gb.ev1));
        if (kernel_ms) *kernel_ms = ms;
    });
}

}  // extern "C"
