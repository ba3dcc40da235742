// The library's one instance of the segmented radix sort (its code object is most of the
// library's size and is loaded at first use: a second instance beside the bit matrix's cost
// the first graph made resident in a process 7 ms).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace blest {

// Scratch bytes for up to `items` keys in up to `segments` segments.
size_t segmented_sort_bytes(uint32_t items, uint32_t segments, int bits, hipStream_t st);
// Sorts the keys of each segment [off[s], off[s + 1]) by their low `bits` bits, ascending.
void segmented_sort(void* temp, size_t bytes, const uint32_t* in, uint32_t* out, uint32_t items, uint32_t segments,
                    const uint32_t* off, int bits, hipStream_t st);

}  // namespace blest
