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

// The shape of a workgroup's work.
enum class FfnShape {
    kSplit,  // up to 32 rows against 64 weight rows, a quarter of k a wave (k_ffn_split)
    kTile,   // one row tile, up to 64 rows, against 256 weight rows, 4-bit codes; three workgroups a compute unit
    kDeep,   // the same with more groups on their way; two workgroups a compute unit
    kWide,   // two row tiles of one expert, up to 128 rows, against 256 weight rows; two workgroups a compute unit
    kLines,  // kDeep for 8-bit codes that are read once: whole 128-byte lines of them, past the caches
};

// The shape of the routed products, from what the host knows (and what a call over a range of the pairs shares with the call
// over all of them: their outputs are the same bytes).
//  - kSplit up to 1,024 pieces of its gate/up launch, two for each of the 512 workgroups it keeps: with 16 experts of
//    1,536 x 1,024 it takes 21 us for 16 tokens where one row tile a workgroup takes 30, and 24.6 against 37.9 for 100 (8-bit
//    codes). Past that it loses: its pieces are short and none of them overlaps the next in its workgroup (256 experts of 2,048
//    x 512, 128 tokens: 150 against 126 us).
//  - kWide where the experts' rows fill its tiles and its launch still has several workgroups for every compute unit; its loop
//    is the most products an unpacked code, its start and end the longest, so k must not be short. kWide against kTile or
//    kDeep, us (pairs an expert; row tiles by column blocks of the gate/up launch):
//      8 bits   256 experts of 2,304 x 1,024: 447, 442 (44; 1,368), 502, 613 (62; 2,000); 32 of 2,880 x 2,880: 294, 315 (62; 713);
//               128 of 1,024 x 512: 73, 81 (70; 560); 100 of 1,024 x 512, uneven: 55, 57 (80; 500); 64 of 2,048 x 512: 92, 92 (87; 348);
//               32 of 1,024 x 1,024: 55, 48 (75; 296); 64 of 512 x 256: 67, 60 (500; 1,000)
//      4 bits, kWide against the better of the others, even and uneven experts (pairs an expert; workgroups times groups of both k):
//               64 of 1,088 x 1,664: 108, 117 and 107, 93 (79; 44 k); 128 of 2,048 x 768: 162, 175 and 167, 155 (75; 40 k); 256 of
//               2,048 x 512: 189, 199 and 162, 154 (62; 40 k), 232, 258 and 216, 212 (94; 60 k); 48 of 3,072 x 1,536, uneven: 182, 188
//               (75; 49 k); 256 of 1,536 x 1,280, uneven: 255, 257 (62; 110 k); 32 of 2,880 x 2,880: 183, 173 (50; 52 k), 210, 222 (62;
//               65 k), 219, 259 (87; 89 k). The line lies where uneven experts stop losing; even ones give 5 to 8 % away below it, and
//               the host cannot tell which it has. With long products the two sides are close up to the line's 56 pairs an expert:
//               256 of 2,304 x 1,024, even, 44, 50, 56 and 62 pairs: 329, 326; 347, 343; 357, 363; 387, 428, uneven 257, 267; 284, 293;
//               304, 318; 332, 346; 64 of 2,880 x 2,048 217, 222; 249, 260; 249, 261; 259, 292, uneven 244, 241; 251, 253; 262, 278; 280, 293.
//  - kTile for 4-bit codes but for the longest k, kDeep for the others. kTile's third workgroup a compute unit hides the start and
//    the end of the short ones, kDeep's loads start earlier: 32 experts of 2,880 x 2,880, 400 tokens 186 against 173 us; 128 of 3,072 x
//    768, 512 uneven tokens 107 against 113; 48 of 3,072 x 1,536, 900 uneven ones 188 against 199, 64 of 1,280 x 2,048, 700 even ones
//    106 against 104, uneven 91 against 95; 256 of 2,048 x 512, 512 uneven ones (129 tiles of 64 rows: more workgroups than kDeep
//    has places for) 71 against 76. Three workgroups with 8-bit codes leave their loads one group ahead: 256 experts of 2,304 x
//    1,024, 1,000 tokens 469 against 439. Some uneven 8-bit chunks miss the third workgroup, others gain, and no size that the host
//    knows tells them apart: whole passes, three workgroups (the loop not yet a pipeline) against kDeep, 128 of 1,536 x 768, 700
//    tokens 115, 123; 128 of 832 x 1,408, 479 tokens 84, 89; 128 of 1,024 x 512, 800 tokens 70, 72; 100 of 1,280 x 1,024, 500
//    tokens 124, 124; 64 of 1,024 x 1,024, 500 tokens 68, 66; 200 of 1,024 x 1,024, 800 tokens 90, 87.
inline FfnShape routed_shape(uint64_t pairs, uint32_t experts, uint32_t d, uint32_t f, uint32_t bits) {
    const uint64_t most_tiles = std::min(pairs, uint64_t(experts)) + pairs / kRowTile;
    if (most_tiles * (f / 32u) <= 1024u) return FfnShape::kSplit;
    const uint64_t workgroups = pairs / kRowTile * ((f + 127u) / 128u);
    if (bits == 8 ? pairs >= 48u * uint64_t(experts) && workgroups >= 450u && d + f >= 1536u
                  : pairs >= 56u * uint64_t(experts) && workgroups * ((d + f) / 64u) >= 46000u && d + f >= 2048u)
        return FfnShape::kWide;
    return bits == 4 && d + f < 5120u ? FfnShape::kTile : FfnShape::kDeep;
}
// ... and of a dense expert's, whose rows are its tiles: kSplit up to two pieces a workgroup (2,048 x 512, 4-bit: 13 against
// 45 us for 37 rows, 16 against 48 for 512, 32 against 47 for 1,500; 2,304 x 1,024, 8-bit: 44 against 54 for 1,000), kDeep
// past that (57 against 79 us for 4,096 rows).
inline FfnShape dense_shape(uint64_t rows, uint32_t f) {
    return (rows + 31u) / 32u * (f / 32u) <= 1024u ? FfnShape::kSplit : FfnShape::kDeep;
}

// The bytes of an expert's codes, scales and biases, wherever its cell lies.
constexpr uint64_t expert_bytes(uint32_t d, uint32_t f, uint32_t bits) { return 3ull * d * f * bits / 8u + 3ull * d * f / 64u * 4u; }

// Whether that many experts are more than the memory-side cache (256 MB) holds, with an eighth to spare: what passes
// by the caches is then nothing that the next pass would have found there. Whole passes over one pool again and again, 8-bit, kDeep
// against non-temporal lines, us: in use 108 MB 85, 91 (128 experts of 832 x 1,408, uneven); 214 MB 72, 77 (128 of 1,024 x 512);
// 267 MB 115, 116 (256 of 2,048 x 512, uneven); 321 MB 93, 86 (48 of 2,048 x 1,024); 369 MB 142, 127 (64 of 1,088 x 1,664); 428 MB
// 113, 106 (128 of 1,024 x 1,024); 820 MB 341, 310 (256 of 2,304 x 1,024, uneven); 1.9 GB 467, 415 (even).
constexpr bool past_the_cache(uint64_t experts, uint32_t d, uint32_t f, uint32_t bits) { return experts * expert_bytes(d, f, bits) >= 288ull << 20; }

// kLines in kDeep's place, where the rows are whole lines from their first byte (`align`: all that a row's address is made of, or-ed)
// and the experts that may be in use are more than the memory-side cache holds. Where they turn out to be fewer, its loads go
// without the hint, and are as fast as kDeep's. (Rows that lines run across: 128 experts of 1,088 x 576, 500 tokens 85 -> 90 us.)
inline FfnShape lines_shape(FfnShape shape, uint64_t pairs, uint32_t experts, uint32_t d, uint32_t f, uint32_t bits, uint64_t align) {
    return shape == FfnShape::kDeep && bits == 8 && align % 128u == 0 && past_the_cache(std::min(pairs, uint64_t(experts)), d, f, bits)
               ? FfnShape::kLines
               : shape;
}

}  // namespace shrike
