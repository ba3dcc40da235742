// Preparation of the resident CSR on the GPU (current device; every call runs on st and is
// complete on return).  ptr: n + 1 ascending list offsets, idx: the entries.  The calls of
// one graph share a stream: making and destroying one costs 50-140 us, a step of a small
// graph about as much (making 1,000 vertices resident 1,085 -> 850 us).
#pragma once

#include <hip/hip_runtime.h>

#include "../csc.hpp"

namespace blest {

// Whether every stored edge has its reverse (columns sorted); throws
// BLEST_ERR_INVALID_ARGUMENT for an entry that is not below n.  found: room for 3 words.
bool csr_symmetric_on_device(hipStream_t st, const uint32_t* ptr, const uint32_t* idx, uint32_t n, uint32_t nnz,
                             unsigned long long* found);
// Orders every list by degree, highest first, ties by ID; csr: the same lists on the host.
void csr_sort_by_degree(hipStream_t st, const CSC& csr, const uint32_t* ptr, uint32_t* idx);
// probe (nullable): each list's first entry, 0 for an empty one; noIn: bit v of the words
// set where list v is empty.
void csr_marks(hipStream_t st, const uint32_t* ptr, const uint32_t* idx, uint32_t n, uint32_t words,
               uint32_t* probe, unsigned long long* noIn);

}  // namespace blest
