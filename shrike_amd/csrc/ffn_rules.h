// What the host decides for the grouped FFN from the sizes of a call alone. Plain C++, so that tests can ask it too.
#pragma once

#include <algorithm>
#include <cstdint>

namespace shrike {

constexpr uint32_t kRowTile = 64;  // rows per row-tile entry (PrefillGroupedRoutedMoE.groupedRowTile)

// Worst case of row tiles for `pairs` pairs over `experts` experts: every expert may end
// in a partly filled tile.
inline uint32_t max_row_tiles(uint64_t pairs, uint32_t experts) {
    return uint32_t(pairs / kRowTile) + experts;
}

// The tile table's records that a launch may ask for before it knows how many there are: those that the table has room for. The
// caller's bound is a bound of the launch and the workspace, which may serve several chunks; the table need not be as long.
inline uint32_t readable_records(uint32_t bound, uint64_t pairs, uint32_t experts) {
    return std::min(bound, max_row_tiles(pairs, experts));
}

}  // namespace shrike
