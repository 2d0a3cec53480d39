// The LDS of the prefill router's workgroups on the matrix cores, from the sizes of a call alone. Plain C++, so that tests can ask it too.
#pragma once

#include <algorithm>
#include <cstdint>

namespace shrike {

template <int RK>
constexpr int kRouterChunk = RK == 0 ? 8 : RK == 8 ? 16 : 32;  // elements of a 16-byte chunk of a row

template <int RK>
struct LogitsLds {
    static constexpr uint32_t kPieces = kRouterChunk<RK> / 8;            // 16-byte pieces of x a chunk
    static constexpr uint32_t kBlock = (kPieces + 1u) * 1024u;           // four chunks of sixteen tokens and sixteen experts
    static constexpr uint32_t kPlaces = RK == 0 ? 3u : 2u;
    // A unit is a walk's chunks, sixteen of each of the four blocks. 4-bit rows of up to 1,536 have no chunks for the last blocks,
    // which then take no place: four workgroups fit a compute unit up to there, where with places for every block three did (256 rows
    // of 1,024, 1,000 tokens: 22.3 -> 20.7 us, 4,000 72.8 -> 68.9; of 1,536, 4,000 tokens 75.8 -> 72.0).
    static constexpr uint32_t blocks(uint32_t d) { return RK == 4 ? std::min(4u, (d / kRouterChunk<RK> + 15u) / 16u) : 4u; }
    static constexpr uint32_t unit(uint32_t d) { return blocks(d) * kBlock; }
    static constexpr uint32_t eff(uint32_t d) { return kPlaces * unit(d); }  // where the widened effective scales lie
    static constexpr uint32_t bytes(uint32_t d) { return eff(d) + 4u * d + (RK ? 2u * 16u * (d / 64u) * 2u : 0u); }
};

}  // namespace shrike
