// Preparation of the resident CSR on the GPU: the symmetry check of the CSC it comes from,
// its lists ordered by degree, the first probes and the vertices without in-neighbours.
// On the host these were most of a graph's loading time (a binary search per stored edge
// and a comparison sort per list): R-MAT 18 22 + 20 ms of a 46 ms upload, R-MAT 22
// 830 + 420 ms of 1.45 s (16 cores); with these 7.6 and 209 ms, most of it transfers.
#include <hipcub/hipcub.hpp>

#include "csr_build.hpp"
#include "scratch.hpp"
#include "segmented_sort.hpp"

namespace blest {
namespace dev {

constexpr int kCsrBlock = 256;
constexpr uint32_t kTileEntries = 4096;  // stored edges a workgroup checks

// Largest c in [lo, hi] with ptr[c] <= p (ptr ascending, ptr[lo] <= p): the column that
// holds entry p, empty columns before it skipped.
__device__ __forceinline__ uint32_t column_of(const uint32_t* ptr, uint32_t lo, uint32_t hi, uint32_t p) {
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (ptr[mid] <= p) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// found[0] |= 1 where an edge j -> i has no edge i -> j (columns sorted), 2 where a row is
// out of range.  A thread takes entries a workgroup apart, so a hub's list is spread over
// workgroups; the columns of a tile are bounded once and searched between the bounds.
// Bound by the dependent reads of the searches.  Half: only the entries whose column i is
// the smaller one (fewer entries, then lower ID) are looked up, in that shorter list;
// found[1] and found[2] count them and the others.  Entries ascending, each entry looked up
// and present is another one of the second kind, so the graph is symmetric iff all are
// present and the two counts agree.  found[0] |= 4 where a column is not strictly ascending:
// that takes the search of every entry.  R-MAT 18 722 -> 312 us, R-MAT 22 17.7 -> 6.4 ms.
template <bool Half>
__global__ void __launch_bounds__(kCsrBlock) csr_symmetry_kernel(const uint32_t* ptr, const uint32_t* idx, uint32_t n,
                                                                 uint32_t nnz, unsigned long long* found) {
    __shared__ uint32_t bound[2];
    __shared__ unsigned sides[2];
    const uint32_t t0 = blockIdx.x * kTileEntries;  // < nnz
    const uint32_t count = min(kTileEntries, nnz - t0);
    if (threadIdx.x < 2) {
        bound[threadIdx.x] = column_of(ptr, 0, n - 1, threadIdx.x ? t0 + count - 1 : t0);
        sides[threadIdx.x] = 0;
    }
    __syncthreads();
    const uint32_t c0 = bound[0], c1 = bound[1];
    unsigned bad = 0, looked = 0, rest = 0;
    for (uint32_t k = threadIdx.x; k < count; k += kCsrBlock) {
        const uint32_t p = t0 + k, i = idx[p];
        if (i >= n) {
            bad |= 2u;
            continue;
        }
        const uint32_t j = column_of(ptr, c0, c1, p);
        uint32_t lo = ptr[i], hi = ptr[i + 1];
        const uint32_t end = hi;
        if (Half) {
            const uint32_t first = ptr[j], mine = ptr[j + 1] - first;
            if (p > first && idx[p - 1] >= i) bad |= 4u;
            if (i == j) continue;
            if (hi - lo > mine || (hi - lo == mine && i > j)) {
                ++rest;
                continue;
            }
            ++looked;
        } else if (i == j) {
            continue;
        }
        while (lo < hi) {  // first entry of column i that is not below j
            const uint32_t mid = lo + (hi - lo) / 2;
            if (idx[mid] < j) lo = mid + 1;
            else hi = mid;
        }
        if (lo == end || idx[lo] != j) bad |= 1u;
    }
    if (Half) {
        if (looked) atomicAdd(&sides[0], looked);
        if (rest) atomicAdd(&sides[1], rest);
        __syncthreads();
        if (threadIdx.x < 2 && sides[threadIdx.x]) atomicAdd(&found[1 + threadIdx.x], (unsigned long long)sides[threadIdx.x]);
    }
    if (bad) atomicOr(found, (unsigned long long)bad);
}

// Radix keys that put the highest degree first; the sort is stable, so ties stay by ID.
__global__ void csr_degree_keys_kernel(const uint32_t* ptr, uint32_t n, uint32_t* key, uint32_t* id) {
    for (uint64_t v = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; v < n; v += uint64_t(gridDim.x) * kCsrBlock) {
        key[v] = ~(ptr[v + 1] - ptr[v]);
        id[v] = uint32_t(v);
    }
}

__global__ void csr_rank_kernel(const uint32_t* order, uint32_t n, uint32_t* rank) {
    for (uint64_t k = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; k < n; k += uint64_t(gridDim.x) * kCsrBlock) rank[order[k]] = uint32_t(k);
}

__global__ void csr_gather_kernel(const uint32_t* table, const uint32_t* from, uint32_t items, uint32_t* to) {
    for (uint64_t e = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; e < items; e += uint64_t(gridDim.x) * kCsrBlock)
        to[e] = table[from[e]];
}

// off[i] = first entry of column c0 + i relative to the batch (i = 0..cols)
__global__ void csr_offsets_kernel(const uint32_t* ptr, uint32_t c0, uint32_t cols, uint32_t e0, uint32_t* off) {
    for (uint64_t i = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; i <= cols; i += uint64_t(gridDim.x) * kCsrBlock)
        off[i] = ptr[c0 + i] - e0;
}

__global__ void csr_probe_kernel(const uint32_t* ptr, const uint32_t* idx, uint32_t n, uint32_t* probe) {
    for (uint64_t v = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; v < n; v += uint64_t(gridDim.x) * kCsrBlock)
        probe[v] = ptr[v + 1] > ptr[v] ? idx[ptr[v]] : 0u;
}

__global__ void csr_no_in_kernel(const uint32_t* ptr, uint32_t n, uint32_t words, unsigned long long* noIn) {
    for (uint64_t v = blockIdx.x * uint64_t(kCsrBlock) + threadIdx.x; v < uint64_t(words) * 64; v += uint64_t(gridDim.x) * kCsrBlock) {
        const unsigned long long b = __ballot(v < n && ptr[v + 1] == ptr[v]);
        if (lane_id() == 0) noIn[v >> 6] = b;
    }
}

}  // namespace dev

bool csr_symmetric_on_device(hipStream_t st, const uint32_t* ptr, const uint32_t* idx, uint32_t n, uint32_t nnz,
                             unsigned long long* found) {
    if (nnz == 0) return true;
    const StreamDrain drain{st};
    unsigned long long got[3] = {0, 0, 0};
    const auto check = [&](auto kernel) {
        got[0] = got[1] = got[2] = 0;
        BLEST_HIP(hipMemcpyAsync(found, got, sizeof(got), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(kernel, dim3((nnz - 1) / dev::kTileEntries + 1), dim3(dev::kCsrBlock), 0, st, ptr, idx, n,
                           nnz, found);
        BLEST_HIP(hipGetLastError());
        BLEST_HIP(hipMemcpyAsync(got, found, sizeof(got), hipMemcpyDeviceToHost, st));
        BLEST_HIP(hipStreamSynchronize(st));
        if (got[0] & 2u) throw Error(BLEST_ERR_INVALID_ARGUMENT, "row index out of range");
    };
    check(dev::csr_symmetry_kernel<true>);
    if (got[0] & 4u) check(dev::csr_symmetry_kernel<false>);
    return got[0] == 0 && got[1] == got[2];
}

void csr_sort_by_degree(hipStream_t st, const CSC& csr, const uint32_t* ptr, uint32_t* idx) {
    const uint32_t n = csr.n;
    // column batches of at most 2^28 entries (one column may exceed that alone)
    constexpr uint64_t kBatch = uint64_t(1) << 28;
    std::vector<uint32_t> cuts{0};
    uint64_t maxItems = 1, maxCols = 1;
    while (cuts.back() < n) {
        const uint32_t c0 = cuts.back();
        const auto from = csr.colPtrs.begin() + c0;
        const uint64_t limit = uint64_t(*from) + kBatch;
        uint32_t c1 = uint32_t(std::upper_bound(from, csr.colPtrs.end(), limit,
                                                [](uint64_t l, uint32_t x) { return l < x; }) - csr.colPtrs.begin()) - 1;
        c1 = std::min(n, std::max(c1, c0 + 1));
        maxItems = std::max<uint64_t>(maxItems, csr.colPtrs[c1] - csr.colPtrs[c0]);
        maxCols = std::max<uint64_t>(maxCols, c1 - c0);
        cuts.push_back(c1);
    }
    if (maxItems > 0x7FFFFFFFull || n > 0x7FFFFFFFu) throw Error(BLEST_ERR_UNSUPPORTED, "list too long for a device sort");
    Scratch sc;
    const StreamDrain drain{st};
    uint32_t* order = sc.alloc<uint32_t>(n);
    uint32_t* rank = sc.alloc<uint32_t>(n);
    uint32_t* keysIn = sc.alloc<uint32_t>(std::max<uint64_t>(maxItems, n));
    uint32_t* keysOut = sc.alloc<uint32_t>(std::max<uint64_t>(maxItems, n));
    uint32_t* off = sc.alloc<uint32_t>(maxCols + 1);
    int bits = 1;
    while ((uint64_t(1) << bits) < n) ++bits;
    size_t pairBytes = 0;
    const size_t segBytes = segmented_sort_bytes(uint32_t(maxItems), uint32_t(maxCols), bits, st);
    BLEST_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, pairBytes, keysIn, keysOut, rank, order, int(n), 0, 32, st));
    void* temp = sc.alloc<uint8_t>(std::max(pairBytes, segBytes));
    const dim3 block(dev::kCsrBlock);
    hipLaunchKernelGGL(dev::csr_degree_keys_kernel, grid_for(n), block, 0, st, ptr, n, keysIn, rank);
    BLEST_HIP(hipGetLastError());
    BLEST_HIP(hipcub::DeviceRadixSort::SortPairs(temp, pairBytes, keysIn, keysOut, rank, order, int(n), 0, 32, st));
    hipLaunchKernelGGL(dev::csr_rank_kernel, grid_for(n), block, 0, st, order, n, rank);
    BLEST_HIP(hipGetLastError());
    for (size_t k = 0; k + 1 < cuts.size(); ++k) {
        const uint32_t c0 = cuts[k], cols = cuts[k + 1] - c0, e0 = csr.colPtrs[c0];
        const uint32_t items = csr.colPtrs[cuts[k + 1]] - e0;
        if (items == 0) continue;
        hipLaunchKernelGGL(dev::csr_offsets_kernel, grid_for(uint64_t(cols) + 1), block, 0, st, ptr, c0, cols, e0, off);
        hipLaunchKernelGGL(dev::csr_gather_kernel, grid_for(items), block, 0, st, rank, idx + e0, items, keysIn);
        BLEST_HIP(hipGetLastError());
        segmented_sort(temp, segBytes, keysIn, keysOut, items, cols, off, bits, st);
        hipLaunchKernelGGL(dev::csr_gather_kernel, grid_for(items), block, 0, st, order, keysOut, items, idx + e0);
        BLEST_HIP(hipGetLastError());
    }
    BLEST_HIP(hipStreamSynchronize(st));
}

void csr_marks(hipStream_t st, const uint32_t* ptr, const uint32_t* idx, uint32_t n, uint32_t words,
               uint32_t* probe, unsigned long long* noIn) {
    const dim3 block(dev::kCsrBlock);
    if (probe) hipLaunchKernelGGL(dev::csr_probe_kernel, grid_for(n), block, 0, st, ptr, idx, n, probe);
    hipLaunchKernelGGL(dev::csr_no_in_kernel, grid_for(uint64_t(words) * 64), block, 0, st, ptr, n, words, noIn);
    BLEST_HIP(hipGetLastError());
    BLEST_HIP(hipStreamSynchronize(st));
}

}  // namespace blest
