#include "segmented_sort.hpp"

#include <hipcub/hipcub.hpp>

#include "dgraph.hpp"

namespace blest {

size_t segmented_sort_bytes(uint32_t items, uint32_t segments, int bits, hipStream_t st) {
    size_t bytes = 0;
    const uint32_t* in = nullptr;
    uint32_t* out = nullptr;
    const uint32_t* off = nullptr;
    BLEST_HIP(hipcub::DeviceSegmentedRadixSort::SortKeys(nullptr, bytes, in, out, int(items), int(segments), off, off,
                                                         0, bits, st));
    return bytes;
}

void segmented_sort(void* temp, size_t bytes, const uint32_t* in, uint32_t* out, uint32_t items, uint32_t segments,
                    const uint32_t* off, int bits, hipStream_t st) {
    BLEST_HIP(hipcub::DeviceSegmentedRadixSort::SortKeys(temp, bytes, in, out, int(items), int(segments), off, off + 1,
                                                         0, bits, st));
}

}  // namespace blest
