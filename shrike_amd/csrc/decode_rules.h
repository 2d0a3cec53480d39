// What the host decides for the decode launches from the sizes of a call alone. Plain C++, so that tests can ask it too.
#pragma once

#include <cstdint>

namespace shrike {

// steps of a wave, 64 chunks of 16 bytes each, that a row of n codes takes
inline uint32_t nch_for(uint32_t n, uint32_t bits) { return (n * bits / 128u + 63u) / 64u; }

// whether a row of `cpr` 16-byte chunks is walked as cpr / 64 whole steps and a step of half chunks
inline bool half_chunk_tail(uint32_t cpr, uint32_t bits) { return bits == 4u && cpr > 64u && (cpr % 64u) >= 1u && (cpr % 64u) <= 32u; }

// Steps of row pairs that a wave of phase 1's routing launch for several tokens walks: two where the launch of one-step waves has 4,096
// workgroups, 16 a compute unit, or more, else one: with fewer the last waves' second steps cost more than the selections saved.
// A layer with one step and with two, us: 16,384 workgroups (16 tokens of 2,304 x 1,024, 8-bit) 172 and 161; 8,192 (8 of them) 95
// and 89; 6,144 (16 of 1,536 x 768) 67 and 65; 4,096 (16 of 2,048 x 512) 57.5 and 55.5; 2,048 (8 of them) 32.8 and 33.1; 1,024 (16 of
// 1,024 x 256) 17.2 and 18.6. What keeps one step:
//  - rows of four steps a lane (12 tokens of 4,096 x 1,024, 8-bit: 190.5 and 192) and rows with half chunks, where the loop's
//    registers cost the launch a wave a SIMD (16 tokens of 2,880 x 2,880: 141 and 144);
//  - 8-bit rows of two or three steps a lane of which more than half the lanes have the last: they are nearer to the memory's rate than
//    to the vector units'. 16 tokens, f 1,024 (3,072: 768), d 1,088 75, 67; 1,280 91, 84; 1,536 77.6, 76.3; 1,792 112, 113; 1,984
//    124, 127; 2,048 125.5, 128; 2,112 142, 134; 2,560 159, 156; 2,816 130.3, 130.8; 2,944 134.8, 136.4; 3,072 184, 186. (Of one step:
//    512 44.8, 43.5; 768 44.3, 44.5; 832 57.0, 57.2; 1,024 72.4, 71.7 and 66.7, 66.7. 4-bit ones of two whole steps: 3,136 128, 119; 3,840
//    127.4, 126.6; 4,096 105.6, 105.8.)
// Two steps' row pairs divide f, a multiple of 64.
inline uint32_t phase1_row_steps(uint64_t workgroups, uint32_t d, uint32_t bits) {
    const uint32_t cpr = d * bits / 128u, steps = nch_for(d, bits), last = cpr - 64u * (steps - 1u);
    if (workgroups < 4096u || steps >= 4u || half_chunk_tail(cpr, bits)) return 1u;
    return bits == 8u && steps >= 2u && last > 32u ? 1u : 2u;
}

}  // namespace shrike
