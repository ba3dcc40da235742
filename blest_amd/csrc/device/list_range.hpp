// Positions in an adjacency list array of up to 2^32 - 1 entries: next to its end, p + step
// passes 2^32 and compares as a small number, so the walks of a list compare distances to its
// end instead.  (No HIP in here: the host test compiles it as it is.)
#pragma once

#include <stdint.h>

namespace blest {
namespace dev {

// End of the first `most` entries of [p, end) (p <= end): all of them where there are fewer.
constexpr uint32_t part_end(uint32_t p, uint32_t end, uint32_t most) { return end - p > most ? p + most : end; }

// Whether entry p + i is one of [p, end) (p <= end).
constexpr bool in_part(uint32_t p, uint32_t i, uint32_t end) { return i < end - p; }

}  // namespace dev
}  // namespace blest
