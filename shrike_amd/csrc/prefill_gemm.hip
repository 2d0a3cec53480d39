// The grouped expert FFN of prefill for gfx950 (PrefillGroupedRoutedMoE.encodeGroupedExpertGEMMs,
// PrefillGroupedRoutedMoE.swift:925-1126): for every 64-row tile of one expert's pairs,
// act = fp16(glu(gate . X, up . X)) and partial = fp16(down . act), on the matrix cores.
//
// The quantised weights never become fp16 weights. With w = q * s + b per group of 64,
//   sum_k x_k w_k = sum_g s_g (sum_{k in g} x_k q_k) + sum_g b_g (sum_{k in g} x_k),
// the codes enter v_mfma_f32_32x32x16_f16 as they are: a 4- or 8-bit code placed in the low
// bits of an fp16 is the subnormal q * 2^-24, which the matrix core multiplies exactly, so
// the per-group product sum_k x_k q_k comes out of four chained MFMAs in fp32 and is scaled
// by s_g * 2^24 on the vector ALU. The bias term is one more short matrix product between
// the per-row group sums of X (fp32 sums carried as fp16 hi + lo, see k_row_group_sums) and
// the group biases.
//
// Two kernels: k_grouped_ffn gives a workgroup a row tile (or two) and a block of weight rows, k_ffn_split a smaller piece
// whose k its waves share; routed_shape and dense_shape (ffn_rules.h) choose.
#include "decode_launch.h"
#include "prefill_common.h"

#include "../../include/shrike_host.h"

#include <type_traits>

namespace shrike {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---- the LDS of a workgroup of each shape: a ring of places for groups of the rows and one for 64-byte units of the
// codes, that asynchronous loads fill (lane l's piece of a load lands 16 l bytes behind the load's address).
constexpr uint32_t kUnitB = 64u * 64u;  // 64 bytes of codes of a wave's 64 weight rows: two groups at 4 bits, one at 8
constexpr uint32_t kUnitS = 64u * 16u;  // four groups' scales (biases) of those rows, in a 12-byte window each
template <FfnShape S, int BITS>
struct Lds {
    static constexpr bool kIsWide = S == FfnShape::kWide;
    static constexpr bool kIsDeep = S == FfnShape::kDeep || S == FfnShape::kLines;
    static constexpr uint32_t kPlacesA = !kIsDeep ? 2u : BITS == 4 ? 4u : 3u;  // of groups of rows
    static constexpr uint32_t kPlacesB = !kIsDeep || BITS == 4 ? 2u : 3u;      // of units of codes
    static constexpr uint32_t kRows = kIsWide ? 128u : 64u;
    static constexpr uint32_t kUnitA = kRows * 128u;  // one group (64 k) of the rows
    static constexpr uint32_t kB = kPlacesA * kUnitA, kS = kB + kPlacesB * 4u * kUnitB, kDst = kS + 4u * kUnitS, kBytes = kDst + kRows * 8u;
    // two units (32 groups each) of the rows' group sums: where the rows and, this one, the codes of the last place will be
    static constexpr uint32_t kSums1 = kS - 4u * kUnitB;
    static_assert(kUnitA <= 4u * kUnitB, "a unit of sums fits");
    static constexpr uint32_t kRow = 128u + 8u;  // halves per row of activations on the way out; the pad spreads the banks
    static constexpr uint32_t kResident = S == FfnShape::kTile ? 3u : 2u;  // workgroups a compute unit holds
    static_assert(kRows * kRow * 2u <= kBytes && kBytes * kResident <= 160u * 1024u, "the rows on the way out fit, and the workgroups a compute unit");
};
struct SplitLds {  // of a wave: 32 rows' groups, the codes of 64 weight rows, their scales and biases
    static constexpr uint32_t kUnitA = 32u * 128u;
    static constexpr uint32_t kB = 2u * kUnitA, kS = kB + 2u * kUnitB, kBias = kS + kUnitS, kWave = kBias + kUnitS, kBytes = 4u * kWave;
    static_assert(2u * kBytes <= 160u * 1024u && kBytes >= 4u * 32u * 64u * 4u, "two workgroups fit a compute unit, and the partial sums a workgroup");
};
static_assert(kRowTile == 64, "a row tile is one or two 32-row MFMA tiles");
constexpr float kTwo24 = 16777216.0f;

struct FfnArgs {
    PoolArg pool;
    uint64_t stride;
    shrike_expert_offsets off;
    const shrike_row_tile *tiles;
    const uint32_t *tile_count;
    const uint64_t *residency;    // null, or the table that names the tiles' cells at this call
    uint32_t pair_lo, pair_hi;    // the sorted pairs this call covers; rows of other pairs are left alone
    const shrike_token_expert_pair *pairs;
    const uint16_t *hidden;       // fp16[T, hidden_stride]
    uint32_t hidden_stride;
    const uint32_t *hidden_sums;  // (hi, lo)[T, d / 64]
    uint16_t *act;                // fp16[tiles * 64, f]
    const uint32_t *act_sums;     // (hi, lo)[tiles * 64, f / 64]
    uint16_t *partials;           // fp16[T * top_k, d]
    uint32_t d, f, top_k, meta, act_kind, ebias;
    // dense mode (one resident FFN over all rows, the shared expert): the three projections as
    // separate tensors, rows in token order, output row = token
    const uint8_t *dense_w[3];
    const uint16_t *dense_s[3], *dense_b[3];
    uint32_t dense_rows;
    uint32_t round_gate_up;        // gate and up pass through fp16 before the GLU (dequant_int4.metal:206-287)
    const uint16_t *scalar_gate;   // fp16[rows] or null: row m's output * sigmoid(gate[m]) (moe.metal:1195-1207)
    uint32_t table_room;           // records that the tile table has room for
    uint32_t resident_workgroups;  // workgroups of the launched k_grouped_ffn the device holds at once
};

// The sum of a group of 64 fp16 values of which eight neighbouring lanes hold eight each, in every one of them: a lane's
// values in order, then the lanes pairwise (k_row_group_sums' order).
__device__ __forceinline__ float eighth_sum(const uint32_t (&w)[4]) {
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        sum = __fadd_rn(sum, f16_to_f32(uint16_t(w[t])));
        sum = __fadd_rn(sum, f16_to_f32(uint16_t(w[t] >> 16)));
    }
    return butterfly_of_8(sum);
}

// The two fp16 values of a word, added to c in fp32.
__device__ __forceinline__ float dot2_ones(uint32_t w, float c) {
    half2v v, ones = {_Float16(1.0f), _Float16(1.0f)};
    __builtin_memcpy(&v, &w, sizeof v);
    return __builtin_amdgcn_fdot2(v, ones, c, false);
}

union Frag {
    half8 h;
    uint32_t u[4];
    uint4 v;
};

// 4-bit: the eight codes of one word as fp16 subnormals, in order: even and odd codes to a byte each, then pairs of bytes
// spread over the halves of a word.
__device__ __forceinline__ half8 codes4(uint32_t w) {
    const uint32_t even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
    Frag f;
    f.u[0] = __builtin_amdgcn_perm(odd, even, 0x0c040c00u);
    f.u[1] = __builtin_amdgcn_perm(odd, even, 0x0c050c01u);
    f.u[2] = __builtin_amdgcn_perm(odd, even, 0x0c060c02u);
    f.u[3] = __builtin_amdgcn_perm(odd, even, 0x0c070c03u);
    return f.h;
}
// 8-bit: eight codes of two words, in order
__device__ __forceinline__ half8 codes8(uint32_t w0, uint32_t w1) {
    Frag f;
    f.u[0] = __builtin_amdgcn_perm(0u, w0, 0x0c010c00u);
    f.u[1] = __builtin_amdgcn_perm(0u, w0, 0x0c030c02u);
    f.u[2] = __builtin_amdgcn_perm(0u, w1, 0x0c010c00u);
    f.u[3] = __builtin_amdgcn_perm(0u, w1, 0x0c030c02u);
    return f.h;
}

__device__ __forceinline__ void lds_load12(uint32_t lds, const void *p) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx3 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
typedef uint32_t u32x4_by2 __attribute__((ext_vector_type(4), aligned(2)));  // eight 16-bit values, wherever they start

// One row tile (WIDE: or two of an expert) against one block of weight rows, 64 rows of them a wave. MODE 0: 32 gate and
// the same 32 up rows against the gathered token rows, GLU, fp16 activations out. MODE 1: 64 down rows against the
// activations, fp16 partials scattered to (token, rank). MT = the 32-row MFMA tiles, META = the type of the scales and
// biases (SHRIKE_META_*), both template parameters, so that the main loop is straight-line code.
//
// Everything the loop reads comes through LDS by asynchronous loads, a group of 64 k at a time: the rows (shared by the
// waves), and each wave's own codes and scales. (Loaded by the lanes themselves, a lane's sixteen bytes lie a weight row from
// its neighbour's, 64 lines a load.)
//
// A wave's matrix and vector work run beside each other only where neighbouring instructions do not wait for each other. A
// chain of four MFMAs from zero and the scaling of its own sums behind it take 173 cycles a chain with two waves a SIMD, the
// scaling of the chain before between the MFMAs 145, and 131 is the matrix pipe alone; with one wave 238 against 158. So the
// loop is a pipeline: between the MFMAs of chain c stand the scaling of chain c - 1, a share of the next codes' unpacking and
// the reads of the rows that the next chain takes, and the wait for the next group's loads stands two chains ahead of their
// use. What bounds it now: with many rows the power that matrix work, its operands' way through LDS and the loads take
// together (2,048 gpt-oss tokens back to back: the clock at 1.95 GHz of 2.4; the kWide gate/up launch keeps the matrix pipe
// busy 47 % of the cycles, vector issue 45 %); with few rows the weights' bytes (kLines, 8-bit, 1,000 tokens: 4.9 TB/s), and the start and
// the end of the many short workgroups (256 experts of 2,048 x 512, 512 tokens: 29 % of the workgroups' time in gate/up and 53 % in
// down lie outside the loop, 27 of 69 us; 37 tokens: 29 and 56 %). Both products, a chain scaled where it ends ->
// pipelined: 32 experts of 2,880 x 2,880, 4-bit, 2,048 tokens 540 -> 495 us, 300 tokens 179 -> 164; 256 of 2,048 x 512, 4,096
// tokens 316 -> 302, 37 33.5 -> 31.4; 256 of 2,304 x 1,024, 8-bit, 1,000 tokens 469 -> 439, 4,000 735 -> 710.
//
// kLines: what a card's memory gives depends on how it is asked. Read once and non-temporally, in whole 128-byte lines, 1.2 GB come
// at 7.1 TB/s; without the hint at 6.2; in halves of a line, a group of 64 codes a row as the other shapes ask for 8-bit ones, at
// 5.7, and at 4.7 with the hint, which drops a line between its halves. So a unit of codes is a line (two groups) of the rows of one
// of a wave's two tiles, three such places take the room of three half-line ones, and the wave takes a unit into registers as soon
// as it has landed, so that its place is asked for again two groups early. Both products of 1,000 kimi tokens (8-bit): 453 -> 407 us;
// whole passes 551 -> 505 us, of 60 uneven tokens 108 -> 95, 17 tokens of 256 x 2,048 x 512 100 -> 92. What is left: the loads alone
// take 221 of the gate/up launch's 240 us and 97 of down's 137. (Four places for tiles of up to 32 rows 263 -> 257 us, the loads dealt over the
// MFMAs that follow a meeting 260 -> 258, the group sums straight to registers 260 -> 258 and elsewhere slower: taken back. The
// same for 4-bit codes: 1,000 even kimi tokens 352 -> 334 us, uneven ones 264 -> 271, 100 tokens of 256 x 2,048 x 512 137 -> 139.)
//
// MODE 0 leaves its activations through LDS: whole 16-byte pieces of a row go out together, and the group sums of the
// tile's rows that the down product's bias term needs are formed here, in k_row_group_sums' order of additions (eight
// lanes a group, a lane adds its eight values in order, the partial sums fold pairwise), instead of by a launch of
// their own between the two products. Every wave of the workgroup stays to the end for the barriers.
template <int BITS, int MODE, bool DENSE, uint32_t MT, int META, FfnShape S>
__device__ __forceinline__ void ffn_tile(const FfnArgs &a, const shrike_row_tile &tile, uint32_t act_row, uint32_t col_block,
                                         uint8_t *lds, bool once) {
    typedef Lds<S, BITS> L;
    // (kTile's places for up to 64 rows are twice as many for up to 32)
    constexpr bool kHalves = S == FfnShape::kTile && MT == 1u;
    constexpr uint32_t kA = L::kPlacesA * (kHalves ? 2u : 1u), kB = L::kPlacesB, kUnitA = L::kUnitA / (kHalves ? 2u : 1u);
    constexpr uint32_t kSums0 = L::kB - kUnitA;
    constexpr bool kLines = S == FfnShape::kLines;
    static_assert(!kLines || (BITS == 8 && !DENSE && MT <= 2u), "kLines is for 8-bit codes of routed experts");
    const uint32_t K = MODE == 0 ? a.d : a.f, N = MODE == 0 ? a.f : a.d;
    const uint32_t G = K / kGroup;
    const uint32_t lane = threadIdx.x & 63u, wave = wave_index();
    const uint32_t col = lane & 31u, kb = lane >> 5;
    const uint32_t n0 = (col_block * 4u + wave) * (MODE == 0 ? 32u : 64u);
    const bool active = n0 < N;
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)lds));
    uint16_t (*s_out)[L::kRow] = reinterpret_cast<uint16_t (*)[L::kRow]>(lds);

    // ---- A: the tile's rows, a group of them (128 bytes a row) at a time. A load brings eight rows, eight lanes a row, its
    // sixteen-byte pieces xor-ed with half the row's number so that sixteen rows read at one piece touch each of the 64 banks once
    // (and those of the codes below, four a row, with a quarter of it). With the whole of it and half, right for 32 banks, the
    // kWide gate/up launch over 2,048 gpt-oss tokens had conflicts of 25.4 M cycles of the compute units' 170 M, now 4.9 M; both
    // products of 512 tokens, 256 experts of 2,048 x 512, 76.2 -> 74.3 us, long chunks within 1 %.
    constexpr uint32_t kLoadsA = MT;  // a wave's loads a group
    constexpr bool kNear = S != FfnShape::kDeep;  // a row is a 32-bit offset from a base (the launch's rule)
    const uint8_t *a_src[kLoadsA];
    uint32_t a_off[kLoadsA];
    const uint8_t *a_base = MODE == 0 ? reinterpret_cast<const uint8_t *>(a.hidden) : reinterpret_cast<const uint8_t *>(a.act + size_t(act_row) * a.f);
    const uint32_t *a_sums[kLoadsA];  // the rows' group sums, for the bias term
#pragma unroll
    for (uint32_t j = 0; j < kLoadsA; ++j) {
        const uint32_t r = min(8u * (wave + 4u * j) + (lane >> 3), tile.rows - 1u);  // rows past the tile repeat its last row
        const uint16_t *row;
        if (MODE == 0) {
            const uint32_t token = DENSE ? tile.pair_start + r : a.pairs[tile.pair_start + r].token;
            row = a.hidden + size_t(token) * a.hidden_stride;
            a_sums[j] = a.hidden_sums + size_t(token) * G;
        } else {
            row = a.act + (size_t(act_row) + r) * a.f;
            a_sums[j] = a.act_sums + (size_t(act_row) + r) * G;
        }
        a_src[j] = reinterpret_cast<const uint8_t *>(row) + (((lane & 7u) ^ (4u * (wave & 1u) + (lane >> 4))) * 16u);
        if (kNear) a_off[j] = uint32_t(a_src[j] - a_base);
    }
    auto load_a = [&](uint32_t slot, uint32_t g) {
#pragma unroll
        for (uint32_t j = 0; j < kLoadsA; ++j) {
            if (kNear) lds_load16(lds0 + slot * kUnitA + (wave + 4u * j) * 1024u, a_base + size_t(g) * 128u, a_off[j]);
            else lds_load16(lds0 + slot * kUnitA + (wave + 4u * j) * 1024u, a_src[j] + size_t(g) * 128u);
        }
    };

    // ---- B: a wave's own 64 weight rows (two tiles of 32), 64 bytes of each at a time
    const uint8_t *base = DENSE ? nullptr : cell_base_uniform(a.pool, tile.cell, a.stride);
    const uint32_t row_bytes = K * BITS / 8u;
    const uint8_t *w_base[2], *s_base[2];
    const uint16_t *b_base[2];
    // row c of tile nt: MODE 0 the same of gate and up, MODE 1 every second, so that a lane's two sums of a row are neighbours
    auto row_of = [&](uint32_t nt, uint32_t c) -> uint32_t { return min(MODE == 0 ? n0 + c : n0 + 2u * c + nt, N - 1u); };
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        if (DENSE) {
            const int p = MODE == 0 ? nt : 2;
            w_base[nt] = a.dense_w[p];
            s_base[nt] = reinterpret_cast<const uint8_t *>(a.dense_s[p]);
            b_base[nt] = a.dense_b[p];
        } else if (MODE == 0) {
            w_base[nt] = base + (nt ? a.off.up_w_off : a.off.gate_w_off);
            s_base[nt] = base + (nt ? a.off.up_s_off : a.off.gate_s_off);
            b_base[nt] = reinterpret_cast<const uint16_t *>(base + (nt ? a.off.up_b_off : a.off.gate_b_off));
        } else {
            w_base[nt] = base + a.off.down_w_off;
            s_base[nt] = base + a.off.down_s_off;
            b_base[nt] = reinterpret_cast<const uint16_t *>(base + a.off.down_b_off);
        }
    }
    // (rows past the last, of a block's waves that have none, are the last one's: loaded, never multiplied)
    uint32_t b_off[4];
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j)
        b_off[j] = row_of(j >> 1, 16u * (j & 1u) + (lane >> 2)) * row_bytes + ((lane & 3u) ^ (lane >> 4)) * 16u;
    // (at 4 bits a row of an odd number of groups ends halfway through its last stage: the lanes of the missing half take
    // the other half's pieces, so that nothing past a tensor's last row is read)
    const uint32_t half_back = (((lane & 3u) ^ (lane >> 4)) & 2u) * 16u;
    constexpr uint32_t kGroupsPerB = BITS == 4 ? 2u : 1u;
    const uint32_t lds_b = lds0 + L::kB + wave * kUnitB;
    // kLines: a unit is a line, 128 bytes or two groups, of each row of ONE of the wave's tiles; load j brings eight rows of it,
    // eight lanes a row.
    const uint32_t line_row0 = min(n0, N - (MODE == 0 ? 32u : 64u));
    uint32_t line_off[4];
    if constexpr (kLines) {
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j)
            line_off[j] = (line_row0 + (MODE == 0 ? 1u : 2u) * (8u * j + (lane >> 3))) * row_bytes + ((lane & 7u) ^ (4u * (j & 1u) + (lane >> 4))) * 16u;
    }
    auto load_line = [&](uint32_t slot, uint32_t nt, uint32_t unit) {
        const uint8_t *at = w_base[nt] + size_t(unit) * 128u + (MODE == 1 && nt ? row_bytes : 0u);
        auto load = [&](auto once) {
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) lds_load16<decltype(once)::value>(lds_b + slot * (4u * kUnitB) + j * 1024u, at, line_off[j]);
        };
        if (once) load(std::true_type{});
        else load(std::false_type{});
    };
    auto load_b = [&](uint32_t slot, uint32_t stage, bool may_end = true) {
        const uint32_t back = BITS == 4 && may_end && 2u * stage + 1u >= G ? half_back : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) lds_load16(lds_b + slot * (4u * kUnitB) + j * 1024u, w_base[j >> 1] + size_t(stage) * 64u, b_off[j] - back);
    };

    // ---- scales: of four groups at a time, lane l row l of the wave's 64. A row's run of scales is two-byte aligned; what
    // is loaded is the window of three words that holds it, never past the word of the tensor's last scale. `s_at` is where a
    // row's chunk starts, from the word that holds the tensor's start; the run then starts max(s_at & 3, s_at - last window)
    // bytes into the window.
    const uint32_t s_row[2] = {row_of(0, col), row_of(1, col)};
    uint32_t s_at[2], s_last[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const uint32_t skew = uint32_t(reinterpret_cast<uintptr_t>(s_base[nt]) & 3u);
        s_at[nt] = skew + s_row[nt] * G * 2u;
        s_last[nt] = ((skew + N * G * 2u + 3u) & ~3u) - 12u;
    }
    const uint8_t *s_src = kb ? s_base[1] : s_base[0];
    s_src -= reinterpret_cast<uintptr_t>(s_src) & 3u;
    const uint32_t s_mine = kb ? s_at[1] : s_at[0], s_mine_last = kb ? s_last[1] : s_last[0];
    const uint32_t lds_s = lds0 + L::kS + wave * kUnitS;
    auto load_s = [&](uint32_t c) { lds_load12(lds_s, s_src + min((s_mine & ~3u) + 8u * c, s_mine_last)); };

    const uint16_t *bias_row[2] = {b_base[0] + size_t(s_row[0]) * G, b_base[1] + size_t(s_row[1]) * G};
    auto eight_at = [&](const uint16_t *row, uint32_t at) {  // groups min(at, G - 8) ...
        const u32x4_by2 v = *reinterpret_cast<const u32x4_by2 *>(row + min(at, G - 8u));
        return make_uint4(v.x, v.y, v.z, v.w);
    };
    // MODE 1: where the rows go, in bytes from `partials` (all ones: nowhere); a dense expert's rows lie where their tokens do, and
    // have the divisors of their scalar gates there instead, if any
    uint64_t *s_dst = reinterpret_cast<uint64_t *>(lds + L::kDst);
    float *s_gate = reinterpret_cast<float *>(lds + L::kDst);
    uint64_t dst = ~0ull;
    uint16_t gate_bits = 0;
    if (MODE == 1 && threadIdx.x < MT * 32u && threadIdx.x < tile.rows) {
        const uint32_t pair = tile.pair_start + threadIdx.x;
        if (DENSE) {
            if (a.scalar_gate) gate_bits = a.scalar_gate[pair];
        } else if (pair >= a.pair_lo && pair < a.pair_hi) {  // a call over a range of the sorted pairs writes their rows only
            const shrike_token_expert_pair p = a.pairs[pair];
            dst = (uint64_t(p.token) * a.top_k + p.rank) * a.d * 2u;
        }
    }
    // what the first group needs is on its way before anything else
    load_s(0);
    if (kLines) {
        load_line(0, 0, 0);
        load_line(1, 1, 0);
    } else {
        load_b(0, 0);
    }
    load_a(0, 0);
    // (what the first group needs first, then of the rest what fits beside the sums below)
#pragma unroll
    for (uint32_t i = 1; !kLines && i + 1u < kB; ++i)
        if (i * kGroupsPerB < G) load_b(i, i);
#pragma unroll
    for (uint32_t i = 1; i + 1u < kA; ++i)
        if (i < G) load_a(i, i);

    if (MODE == 1 && !DENSE && threadIdx.x < MT * 32u) s_dst[threadIdx.x] = dst;

    // (4-bit codes: the place of the second unit of sums is free where there is none. 128 experts of 2,048 x 1,024, 300 tokens,
    // weights from memory: 124 -> 120 us.)
    const bool last_b_early = BITS == 4 && G <= 32u && (kB - 1u) * kGroupsPerB < G;
    if (last_b_early) load_b(kB - 1u, kB - 1u);

    f32x16 total[2][MT];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (uint32_t mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) total[nt][mt][i] = 0.0f;

    // ---- bias term: (group sums of the rows) x (group biases), sixteen k' = eight groups an MFMA, four of them a lane.
    // The sums come through the LDS like the rows, 32 groups (128 bytes a row) a unit, two units at a time, in the places that
    // the second group's operands will take. A weight row's biases are a lane's own loads, eight groups each; the groups of an
    // MFMA are dealt so that a lane's eight serve two of them. The last eight start at G - 8 at the latest, and what they
    // repeat counts as zero.
    auto bias_f16 = [&](uint16_t bits) { return META == SHRIKE_META_BF16 ? f32_to_f16(bf16_to_f32(bits)) : bits; };
    if (G >= 8u) {
        for (uint32_t g0 = 0; g0 < G; g0 += 64u) {
            if (g0) wait_loads_and_sync<0>();
            // piece q of a unit: the four groups h of lane half k's eight, load i
#pragma unroll
            for (uint32_t u = 0; u < 2u; ++u) {
                if (g0 + 32u * u >= G) break;
                const uint32_t q = (lane & 7u) ^ (lane >> 3);
                const uint32_t at = min(g0 + 32u * u + 16u * (q >> 2) + 8u * ((q >> 1) & 1u), G - 8u) + 4u * (q & 1u);
#pragma unroll
                for (uint32_t j = 0; j < kLoadsA; ++j)
                    lds_load16(lds0 + (u ? L::kSums1 : kSums0) + (wave + 4u * j) * 1024u, a_sums[j] + at);
            }
            uint4 b8[2][2][2];  // [unit][load][nt]
            if (active) {
#pragma unroll
                for (uint32_t u = 0; u < 2u; ++u)
#pragma unroll
                    for (uint32_t i = 0; i < 2u; ++i) {
                        const uint32_t at = g0 + 32u * u + 16u * i;
                        if (at >= G) break;
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt) b8[u][i][nt] = eight_at(bias_row[nt], at + 8u * kb);
                    }
            }
            wait_loads_and_sync<0>();
            if (!active) continue;
#pragma unroll
            for (uint32_t u = 0; u < 2u; ++u)
#pragma unroll
                for (uint32_t i = 0; i < 2u; ++i) {
                    if (g0 + 32u * u + 16u * i >= G) break;
                    const uint32_t at = g0 + 32u * u + 16u * i + 8u * kb, repeated = at - min(at, G - 8u);
#pragma unroll
                    for (uint32_t h = 0; h < 2u; ++h) {
                        const uint8_t *p = lds + (u ? L::kSums1 : kSums0) + col * 128u + (((4u * i + 2u * kb + h) ^ (col & 7u)) * 16u);
                        half8 sums[MT];
#pragma unroll
                        for (uint32_t mt = 0; mt < MT; ++mt) sums[mt] = *reinterpret_cast<const half8 *>(p + mt * 4096u);
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt) {
                            const uint32_t w[4] = {b8[u][i][nt].x, b8[u][i][nt].y, b8[u][i][nt].z, b8[u][i][nt].w};
                            Frag f;
#pragma unroll
                            for (uint32_t jj = 0; jj < 4u; ++jj) {  // as fp16, doubled against (hi, lo)
                                const uint16_t bits = uint16_t(w[2u * h + jj / 2u] >> (16u * (jj & 1u)));
                                f.u[jj] = repeated <= 4u * h + jj ? uint32_t(bias_f16(bits)) * 0x00010001u : 0u;
                            }
#pragma unroll
                            for (uint32_t mt = 0; mt < MT; ++mt) total[nt][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[mt], f.h, total[nt][mt], 0, 0, 0);
                        }
                    }
                }
        }
    } else if (active) {  // fewer than eight groups: one MFMA, value by value
        const uint32_t *sums = MODE == 0 ? a.hidden_sums : a.act_sums;
        Frag afr[MT];
#pragma unroll
        for (uint32_t mt = 0; mt < MT; ++mt) {
            const uint32_t r = min(mt * 32u + col, tile.rows - 1u);
            const uint32_t token = (MODE != 0) ? 0u : DENSE ? tile.pair_start + r : a.pairs[tile.pair_start + r].token;
            const uint32_t *row = MODE == 0 ? sums + size_t(token) * G : sums + (size_t(act_row) + r) * G;
#pragma unroll
            for (uint32_t jj = 0; jj < 4u; ++jj) afr[mt].u[jj] = 4u * kb + jj < G ? row[4u * kb + jj] : 0u;
        }
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            Frag f;
#pragma unroll
            for (uint32_t jj = 0; jj < 4u; ++jj)
                f.u[jj] = 4u * kb + jj < G ? uint32_t(bias_f16(bias_row[nt][4u * kb + jj])) * 0x00010001u : 0u;
#pragma unroll
            for (uint32_t mt = 0; mt < MT; ++mt) total[nt][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(afr[mt].h, f.h, total[nt][mt], 0, 0, 0);
        }
    }

    // ---- the groups: 2 MT chains each, (row tile, weight tile) = (0, 0), (0, 1), (1, 0), ... The fences between the slots
    // keep the order as it is written.
    wait_loads_and_sync<0>();  // (nobody reads the sums any more)
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0) in the compiler's own count: else it waits for the biases in the loop
    // (formed where a sum is written it was a load, expf and a wait a row: 4,096 rows of 2,048 x 512, the down launch 28.8 -> 22.8 us)
    if (MODE == 1 && DENSE && threadIdx.x < MT * 32u) s_gate[threadIdx.x] = 1.0f + expf(-f16_to_f32(gate_bits));
    if (kLines && 2u < G) load_line(2, 0, 1);
    if (!kLines && kA != 2u && !last_b_early && (kB - 1u) * kGroupsPerB < G) load_b(kB - 1u, kB - 1u);
    if (kA - 1u < G) load_a(kA - 1u, kA - 1u);
    if (kA == 2u && !last_b_early && (kB - 1u) * kGroupsPerB < G) load_b(kB - 1u, kB - 1u);
    uint32_t run[2][2];  // the scales of a chunk of four groups, two a word
    float sc[2], sc_before = 0.0f;
    constexpr bool kTwoA = MT <= (S == FfnShape::kTile ? 1u : 2u);  // two sets of a row tile's operands: the next is read a chain earlier
    half8 af[kTwoA ? 2 : 1][4], bf[2][4];
    uint4 raw[kTwoA ? 2 : 1][kLines ? 4 : BITS / 4];
    constexpr bool kBehind = !(S == FfnShape::kTile && MT == 2u);  // (else a chain is scaled where it ends: a third workgroup's waves run beside it)
    f32x16 p[2];
    float tot[2][MT][16];  // (single registers: eight tuples of sixteen beside p do not fit round each other, and two were spilled)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        p[1][i] = 0.0f;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (uint32_t mt = 0; mt < MT; ++mt) tot[nt][mt][i] = total[nt][mt][i];
    }
    auto read_run = [&](uint32_t g) {  // of the chunk that starts at g
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const int into = max(int(s_at[nt] & 3u), int(s_at[nt] + g * 2u) - int(s_last[nt]));
            const uint8_t *q = lds + L::kS + wave * kUnitS + (uint32_t(nt) * 32u + col) * 16u + uint32_t(into);
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (uint32_t i = 0; i < 2u; ++i) {
                u16x2 v;
                v.x = *reinterpret_cast<const uint16_t *>(q + min(2u * i, G - 1u - g) * 2u);
                v.y = *reinterpret_cast<const uint16_t *>(q + min(2u * i + 1u, G - 1u - g) * 2u);
                __builtin_memcpy(&run[nt][i], &v, 4);
            }
        }
    };
    auto next_scales = [&](auto odd) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            sc[nt] = meta_f32(uint16_t(run[nt][0] >> (decltype(odd)::value ? 16 : 0)), uint32_t(META)) * kTwo24;
            if (decltype(odd)::value) run[nt][0] = run[nt][1];
        }
    };
    const uint8_t *a_rows = lds + col * 128u, *b_rows = lds + L::kB + wave * kUnitB + col * 64u;
    auto read_a = [&](uint32_t place, uint32_t mt, uint32_t s) {
        return *reinterpret_cast<const half8 *>(a_rows + place * kUnitA + mt * 4096u + (((kb * 4u + s) ^ ((col >> 1) & 7u)) * 16u));
    };
    auto read_raw = [&](uint32_t nt, uint32_t b_place, uint32_t par) {
#pragma unroll
        for (uint32_t i = 0; i < BITS / 4; ++i) {
            const uint32_t piece = BITS == 4 ? par * 2u + kb : kb * 2u + i;
            raw[kTwoA ? nt : 0u][i] = *reinterpret_cast<const uint4 *>(b_rows + b_place * (4u * kUnitB) + nt * 2048u + ((piece ^ ((col >> 2) & 3u)) * 16u));
        }
    };
    auto read_line = [&](uint32_t slot, uint32_t nt) {
        const uint8_t *p = lds + L::kB + wave * kUnitB + slot * (4u * kUnitB) + col * 128u;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) raw[kTwoA ? nt : 0u][i] = *reinterpret_cast<const uint4 *>(p + (((4u * (i >> 1) + 2u * kb + (i & 1u)) ^ ((col >> 1) & 7u)) * 16u));
    };
    auto unpack = [&](uint32_t nt, uint32_t s, uint32_t par) {
        const uint4 (&codes)[kLines ? 4 : BITS / 4] = raw[kTwoA ? nt : 0u];
        if (kLines) {
            const uint4 v = codes[2u * par + (s >> 1)];
            bf[nt][s] = s & 1u ? codes8(v.z, v.w) : codes8(v.x, v.y);
        } else if (BITS == 4) {
            const uint32_t w[4] = {codes[0].x, codes[0].y, codes[0].z, codes[0].w};
            bf[nt][s] = codes4(w[s]);
        } else {
            const uint4 v = codes[s >> 1 & (BITS / 4 - 1)];
            bf[nt][s] = s & 1u ? codes8(v.z, v.w) : codes8(v.x, v.y);
        }
    };
    // The places of group g's rows and of its codes. Powers of two are known to the compiler four groups at a time.
    uint32_t place3 = 0;  // g % 3
    uint32_t line_at = 0;  // kLines: the place that held the first tile's codes of this unit
    auto next3 = [](uint32_t p) { return p == 2u ? 0u : p + 1u; };
    auto a_place = [&](uint32_t u) { return kA == 3u ? place3 : u & (kA - 1u); };
    auto b_place = [&](uint32_t u) { return kB == 3u ? place3 : BITS == 8 ? u & 1u : (u >> 1) & 1u; };
    // Where group g + 1's operands are all there and the place of group g's rows is free again: what the wave asks for here is
    // for that place. u = g % 4; far: the groups up to the next meeting's g + 4 exist, and which loads may still be on their way
    // is known to the compiler. Else all are waited for, but for 8-bit codes what two more groups need (256 experts of 2,048 x
    // 512, 17 tokens 80.3 -> 79.0 us; at 4 bits the same was nothing or slower).
    auto meet = [&](uint32_t g, auto u_, auto far_) {
        constexpr uint32_t U = decltype(u_)::value;
        constexpr bool FAR = decltype(far_)::value;
        constexpr bool kOdd = (U & 1u) != 0u;
        if constexpr (kLines) {
            constexpr int kLeft = kOdd ? 4 : 8 + int(MT);
            if (FAR || g + (kOdd ? 3u : 2u) < G) wait_loads_and_sync<kLeft>();
            else wait_loads_and_sync<0>();
            if (U == 0u && (FAR || g + 4u < G)) load_s((g >> 2) + 1u);
            if (FAR || g + kA < G) load_a(a_place(U), g + kA);
            if (!kOdd) {
                if (FAR || g + 2u < G) load_line(line_at, 1, (g >> 1) + 1u);
                if (FAR || g + 4u < G) load_line(next3(line_at), 0, (g >> 1) + 2u);
            }
            return;
        }
        // what was asked for at the last meeting, or the last two, and is not needed yet
        constexpr uint32_t kOnTheWay = kA == 2u              ? (BITS == 4 && !kOdd ? 4u : 0u)
                                       : kA == 3u            ? MT + 4u + (U == 1u ? 1u : 0u)
                                       : kOdd                ? 2u * MT + (U == 1u ? 1u : 0u)
                                                             : 2u * MT + 4u + (U == 2u ? 1u : 0u);
        if constexpr (!FAR && kA == 3u) {
            if (g + 2u < G) wait_loads_and_sync<MT + 4>();
            else wait_loads_and_sync<0>();
        } else {
            if (kA == 2u && BITS == 4 && FAR && U == 0u && g == 0u) wait_loads_and_sync<0>();  // (the codes may have been asked for ahead of the rows)
            else wait_loads_and_sync<FAR ? int(kOnTheWay) : 0>();
        }
        if (U == 0u && (FAR || g + 4u < G)) load_s((g >> 2) + 1u);
        if (kA == 2u && (FAR || g + kA < G)) load_a(a_place(U), g + kA);
        if (BITS == 8 && (FAR || g + kB < G)) load_b(b_place(U), g + kB);
        if (BITS == 4 && kOdd && (FAR || g - 1u + 2u * kB < G)) load_b(b_place(U), (g >> 1) + kB, !FAR);
        if (kA != 2u && (FAR || g + kA < G)) load_a(a_place(U), g + kA);
    };
    auto step = [&](uint32_t g, auto u_, auto far_) {
        constexpr uint32_t U = decltype(u_)::value;
        if (!active) {
            meet(g, u_, far_);
            if (kA == 3u) place3 = next3(place3);
            if (kLines && (U & 1u)) line_at = next3(next3(line_at));
            return;
        }
        const uint32_t a_here = a_place(U), a_next = kA == 3u ? next3(place3) : a_place(U + 1u), b_next = kB == 3u ? a_next : b_place(U + 1u);
#pragma unroll
        for (uint32_t c = 0; c < 2u * MT; ++c) {
            const uint32_t mt = c >> 1, nt = c & 1u;
            const uint32_t set = kTwoA ? (U * MT + mt) & 1u : 0u;
            if (c == 2u * MT - 2u) {
                meet(g, u_, far_);
                if (kLines && (U & 1u)) read_line(next3(next3(line_at)), 0);
                if (!kLines) read_raw(0, b_next, (U & 1u) ^ 1u);
                if (U == 3u && (decltype(far_)::value || g + 1u < G)) read_run(g + 1u);
            }
            f32x16 &cur = p[kBehind ? nt : 0u], &old = p[kBehind ? nt ^ 1u : 0u];
            float (&into)[16] = tot[nt ^ 1u][c ? (c - 1u) >> 1 : MT - 1u];
            const float scale = c ? sc[nt ^ 1u] : sc_before;
#pragma unroll
            for (uint32_t s = 0; s < 4u; ++s) {
                f32x16 zero = {0};
                cur = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[set][s], bf[nt][s], s ? cur : zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (nt == (kTwoA ? 0u : 1u)) af[kTwoA ? set ^ 1u : 0u][s] = mt + 1u < MT ? read_a(a_here, mt + 1u, s) : read_a(a_next, 0u, s);
                if (c == 0u) unpack(1, s, U & 1u);
                if (c == 2u * MT - 1u) unpack(0, s, (U & 1u) ^ 1u);
                if (c == 2u * MT - 1u && s == (kTwoA ? 0u : 3u)) {
                    if (kLines && (U & 1u)) read_line(line_at, 1);
                    if (!kLines) read_raw(1, b_next, (U & 1u) ^ 1u);
                }
#pragma unroll
                for (uint32_t i = 4u * s; kBehind && i < 4u * s + 4u; ++i) into[i] = fmaf(scale, old[i], into[i]);
                // (named here: else the additions sink past the branches of `meet`, and every chain's sums stay alive until there)
                if (kBehind) asm volatile("" : "+v"(into[4u * s]), "+v"(into[4u * s + 1u]), "+v"(into[4u * s + 2u]), "+v"(into[4u * s + 3u]));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!kBehind) {
#pragma unroll
                for (uint32_t i = 0; i < 16u; ++i) tot[nt][mt][i] = fmaf(sc[nt], cur[i], tot[nt][mt][i]);
#pragma unroll
                for (uint32_t i = 0; i < 16u; i += 4u) asm volatile("" : "+v"(tot[nt][mt][i]), "+v"(tot[nt][mt][i + 1u]), "+v"(tot[nt][mt][i + 2u]), "+v"(tot[nt][mt][i + 3u]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (kA == 3u) place3 = a_next;
        if (kLines && (U & 1u)) line_at = next3(next3(line_at));
        sc_before = sc[1];
        next_scales(std::integral_constant<bool, (U & 1u) == 0u>{});
    };
    if (active) {
        read_run(0);
        next_scales(std::false_type{});
        if (kLines) read_line(0, 0);
        else read_raw(0, 0, 0);
#pragma unroll
        for (uint32_t s = 0; s < 4u; ++s) {
            af[0][s] = read_a(0, 0, s);
            unpack(0, s, 0);
        }
        if (kLines) read_line(1, 1);
        else read_raw(1, 0, 0);
    }
    uint32_t g = 0;
    for (; g + 8u <= G; g += 4u) {
        step(g, std::integral_constant<uint32_t, 0>{}, std::true_type{});
        step(g + 1u, std::integral_constant<uint32_t, 1>{}, std::true_type{});
        step(g + 2u, std::integral_constant<uint32_t, 2>{}, std::true_type{});
        step(g + 3u, std::integral_constant<uint32_t, 3>{}, std::true_type{});
    }
    for (; g < G; g += 4u) {
        step(g, std::integral_constant<uint32_t, 0>{}, std::false_type{});
        if (g + 1u < G) step(g + 1u, std::integral_constant<uint32_t, 1>{}, std::false_type{});
        if (g + 2u < G) step(g + 2u, std::integral_constant<uint32_t, 2>{}, std::false_type{});
        if (g + 3u < G) step(g + 3u, std::integral_constant<uint32_t, 3>{}, std::false_type{});
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (kBehind) tot[1][MT - 1u][i] = fmaf(sc_before, p[1][i], tot[1][MT - 1u][i]);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (uint32_t mt = 0; mt < MT; ++mt) total[nt][mt][i] = tot[nt][mt][i];
    }
    if (MODE == 0) wait_loads_and_sync<0>();  // (nobody reads the rings any more: the LDS takes the rows on their way out)

    // ---- epilogue: lane holds (m = 32 mt + 8 (i / 4) + 4 kb + i % 4, n = n0 + col)
    const uint32_t n = n0 + col;
    if (MODE == 0) {
        // the tile's fp16 activations, [row][column of this block of 128]
        if (active) {
            float gab = 0.0f, uab = 0.0f;
            if (!DENSE && a.ebias) {  // moe.metal:261-269
                gab = bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.gate_ab_off)[n]);
                uab = bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.up_ab_off)[n]);
            }
            auto activate = [&](auto act) {  // (the choice of the activation is outside the loop)
#pragma unroll
                for (uint32_t mt = 0; mt < MT; ++mt) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const uint32_t m = mt * 32u + 8u * (i / 4) + 4u * kb + (i % 4);
                        float g = total[0][mt][i] + gab, u = total[1][mt][i] + uab;
                        if (DENSE && a.round_gate_up) {
                            g = f16_to_f32(f32_to_f16(g));
                            u = f16_to_f32(f32_to_f16(u));
                        }
                        s_out[m][wave * 32u + col] = f32_to_f16(glu_fast<decltype(act)::value>(g, u));
                    }
                }
            };
            if (a.act_kind == SHRIKE_ACT_SILU) activate(std::integral_constant<int, 1>{});
            else if (a.act_kind == SHRIKE_ACT_CLAMPED_SWIGLU) activate(std::integral_constant<int, 2>{});
            else activate(std::integral_constant<int, 0>{});
        }
        __syncthreads();
        const uint32_t c0 = col_block * 128u, columns = min(128u, N - c0);  // N is a multiple of 64
        // a thread takes an eighth of a (row, group): eight neighbouring columns, out as they are and into the group's sum
        uint32_t *sums_out = const_cast<uint32_t *>(a.act_sums);
#pragma unroll
        for (uint32_t i = 0; i < MT * 2u; ++i) {
            const uint32_t slot = threadIdx.x + 256u * i, m = slot >> 4, gl = (slot >> 3) & 1u, eighth = slot & 7u;
            const uint4 v = *reinterpret_cast<const uint4 *>(&s_out[m][gl * 64u + eighth * 8u]);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
            const float sum = eighth_sum(w);
            if (m < tile.rows && gl * 64u < columns) {
                *reinterpret_cast<uint4 *>(a.act + (size_t(act_row) + m) * a.f + c0 + gl * 64u + eighth * 8u) = v;
                if (eighth == 0u) sums_out[(size_t(act_row) + m) * (a.f / kGroup) + c0 / kGroup + gl] = split_hi_lo(sum);
            }
        }
    } else {
        // a lane's two sums of a row are neighbours: a row's 64 columns of the wave leave as one run of 128 bytes
        if (active) {
            const uint32_t n2 = n0 + 2u * col;
            float dab[2] = {0.0f, 0.0f};
            if (!DENSE && a.ebias) {
                dab[0] = bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.down_ab_off)[n2]);
                dab[1] = bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.down_ab_off)[n2 + 1u]);
            }
            uint8_t *out = reinterpret_cast<uint8_t *>(a.partials) + n2 * 2u;
#pragma unroll
            for (uint32_t mt = 0; mt < MT; ++mt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t m = mt * 32u + 8u * (i / 4) + 4u * kb + (i % 4);
                    const uint64_t to = !DENSE ? s_dst[m] : m < tile.rows ? uint64_t(tile.pair_start + m) * a.d * 2u : ~0ull;
                    uint16_t y0 = f32_to_f16(total[0][mt][i] + dab[0]), y1 = f32_to_f16(total[1][mt][i] + dab[1]);
                    if (DENSE && a.scalar_gate) {  // one gate a token row (moe.metal:1195-1207)
                        const float gate_mul = s_gate[m];
                        y0 = f32_to_f16(f16_to_f32(y0) / gate_mul);
                        y1 = f32_to_f16(f16_to_f32(y1) / gate_mul);
                    }
                    if (to != ~0ull) *reinterpret_cast<uint32_t *>(out + to) = uint32_t(y0) | uint32_t(y1) << 16;
                }
            }
        }
    }
}

template <int BITS, int MODE, bool DENSE, int META, FfnShape S>
__global__ __launch_bounds__(256, (Lds<S, BITS>::kResident)) void k_grouped_ffn(FfnArgs a) {
    warm_kernel_arguments(a);
    __shared__ __align__(16) uint8_t lds[Lds<S, BITS>::kBytes];
    constexpr bool WIDE = S == FfnShape::kWide;
    // Which (row tile, column block) this workgroup takes. Workgroups go to the chip's eight XCDs (each
    // with an L2 of its own) round robin in launch order, so workgroup w runs on XCD w % 8 as that XCD's
    // item w / 8. An expert's row tiles are neighbours in the tile table: an XCD takes a contiguous run
    // of tiles with all their column blocks, so that the column blocks of a tile find its gathered rows,
    // and the row tiles of an expert its codes, in the L2 that fetched them first.
    const uint32_t column_blocks = gridDim.y;
    // (The records of a table of up to 256 tiles, asked for beside the count and not behind it, as far as the table has room: both
    // products of 37 tokens, 256 experts of 2,048 x 512, 32.1 -> 31.5 us, of 512 tokens 76.9 -> 76.4. Four named ones, not an
    // array: the compiler kept an array of them in private memory.)
    const uint32_t lane = threadIdx.x & 63u;
    const uint4 *table = reinterpret_cast<const uint4 *>(a.tiles);
    uint4 rec0 = zero4(), rec1 = zero4(), rec2 = zero4(), rec3 = zero4();
    if (!WIDE && !DENSE) {
        const uint32_t last = a.table_room - 1u;
        rec0 = table[min(lane, last)];
        rec1 = table[min(lane + 64u, last)];
        rec2 = table[min(lane + 128u, last)];
        rec3 = table[min(lane + 192u, last)];
    }
    const uint32_t tile_total = DENSE ? (a.dense_rows + kRowTile - 1u) / kRowTile : *a.tile_count;
    const uint32_t w = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t xcd = w & 7u, item = w >> 3;
    // Where the table is short (64 tiles: one record a lane) and the chip holds the whole launch at once even so, what a tile
    // has past 32 rows is a workgroup's of its own, behind the others. Such a launch is as long as its longest workgroup, and
    // one of more than 32 rows has twice the matrix work a group of k. Measured, both products: 37 tokens of the 35B shape, 38
    // tiles, 45.9 -> 34.8 us; 64 tokens, 49 tiles, 48.3 -> 37.2. Where not every part finds a place at once the codes would be
    // read and converted twice for nothing, so the tiles stay whole. A row's result does not depend on its place in a tile.
    uint32_t parts = tile_total;
    uint64_t larger = 0;
    if (!WIDE && !DENSE && tile_total <= 64u) {
        larger = __ballot(lane < tile_total && rec0.z > 32u);
        parts += uint32_t(__popcll(larger));
        if (parts * column_blocks > a.resident_workgroups || parts + 7u > gridDim.x) {
            parts = tile_total;
            larger = 0;
        }
    }
    // tiles an XCD takes: an eighth of them, the first (total mod 8) XCDs one more
    const uint32_t run = parts / 8u + (xcd < parts % 8u ? 1u : 0u), first = xcd * (parts / 8u) + min(xcd, parts % 8u);
    const uint32_t place = item / column_blocks, col_block = item % column_blocks;  // the workgroup's place in its XCD's run
    if (place >= run) return;
    uint32_t tile_index = first + place, skip = 0;
    shrike_row_tile tile;
    if (DENSE) {
        if (tile_index >= tile_total) return;
        tile.cell = 0;
        tile.pair_start = tile_index * kRowTile;
        tile.rows = min(kRowTile, a.dense_rows - tile.pair_start);
        tile.expert = 0;
    } else {
        if (tile_index >= parts) return;
        // Which tile of the table the workgroup takes. A compute unit holds several of these workgroups, whose waves share its
        // SIMDs' issue, and an XCD's workgroups reach its compute units in launch order, one each before any gets a second
        // (read from the hardware: item i and item i + 32 of an XCD share a unit). A tile of more than 32 rows is twice a
        // smaller one's matrix work, and the launch ends with the units that hold more than one of those.
        //  - Where the gate/up launch fits the chip at once: every XCD takes the same number of the larger tiles (a block of
        //    them in table order, so an expert's stay together) and fills its eighth with a block of the smaller ones; the
        //    larger go first, so each gets a smaller neighbour.
        //  - Otherwise the XCD's eighth is a contiguous run of the table, its larger tiles first: the workgroups that start
        //    late are then the short ones, on the XCDs with the least work.
        // A lane reads one record; the chosen one is read across (no second load).
        const uint32_t gate_up_blocks = (a.f + 127u) / 128u;
        bool chosen = larger != 0u;
        if (chosen) {
            if (tile_index >= tile_total) {
                uint64_t rest = larger;
                for (uint32_t n = tile_index - tile_total; n != 0u; --n) rest &= rest - 1u;
                tile_index = uint32_t(__ffsll((long long)rest)) - 1u;
                skip = 32u;
            }
            tile.cell = uint32_t(__builtin_amdgcn_readlane(int(rec0.x), int(tile_index)));
            tile.pair_start = uint32_t(__builtin_amdgcn_readlane(int(rec0.y), int(tile_index))) + skip;
            const uint32_t rows = uint32_t(__builtin_amdgcn_readlane(int(rec0.z), int(tile_index)));
            tile.rows = skip ? rows - 32u : min(rows, 32u);
            tile.expert = uint32_t(__builtin_amdgcn_readlane(int(rec0.w), int(tile_index)));
        } else if (!WIDE && tile_total <= 256u && tile_total * gate_up_blocks <= a.resident_workgroups) {
            const bool in0 = lane < tile_total, in1 = lane + 64u < tile_total, in2 = lane + 128u < tile_total, in3 = lane + 192u < tile_total;
            const uint64_t larger0 = __ballot(in0 && rec0.z > 32u), larger1 = __ballot(in1 && rec1.z > 32u);
            const uint64_t larger2 = __ballot(in2 && rec2.z > 32u), larger3 = __ballot(in3 && rec3.z > 32u);
            const uint64_t smaller0 = __ballot(in0 && rec0.z <= 32u), smaller1 = __ballot(in1 && rec1.z <= 32u);
            const uint64_t smaller2 = __ballot(in2 && rec2.z <= 32u), smaller3 = __ballot(in3 && rec3.z <= 32u);
            const uint32_t larger_total = uint32_t(__popcll(larger0) + __popcll(larger1) + __popcll(larger2) + __popcll(larger3));
            const uint32_t lq = larger_total / 8u, lr = larger_total % 8u;
            if (lq + 1u <= tile_total / 8u) {  // every XCD's share of the larger tiles fits its eighth
                const uint32_t mine_larger = lq + (xcd < lr ? 1u : 0u), larger_first = xcd * lq + min(xcd, lr);
                const bool take_larger = place < mine_larger;
                uint32_t want = take_larger ? larger_first + place : (first - larger_first) + (place - mine_larger);
                const uint64_t m0 = take_larger ? larger0 : smaller0, m1 = take_larger ? larger1 : smaller1;
                const uint64_t m2 = take_larger ? larger2 : smaller2, m3 = take_larger ? larger3 : smaller3;
                const uint32_t c0 = uint32_t(__popcll(m0)), c1 = uint32_t(__popcll(m1)), c2 = uint32_t(__popcll(m2));
                uint64_t set;
                uint32_t block;
                if (want < c0) { set = m0; block = 0; }
                else if (want < c0 + c1) { set = m1; block = 1; want -= c0; }
                else if (want < c0 + c1 + c2) { set = m2; block = 2; want -= c0 + c1; }
                else { set = m3; block = 3; want -= c0 + c1 + c2; }
                chosen = want < uint32_t(__popcll(set));
                if (chosen) {
                    const bool me = ((set >> lane) & 1ull) != 0ull && uint32_t(__popcll(set & ((1ull << lane) - 1ull))) == want;
                    const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(me)) - 1);
                    auto take = [&](const uint4 &r) {  // (a branch a block, uniform: a select between the four records became an
                                                       // indexed load from private memory)
                        tile.cell = uint32_t(__builtin_amdgcn_readlane(int(r.x), src));
                        tile.pair_start = uint32_t(__builtin_amdgcn_readlane(int(r.y), src));
                        tile.rows = uint32_t(__builtin_amdgcn_readlane(int(r.z), src));
                        tile.expert = uint32_t(__builtin_amdgcn_readlane(int(r.w), src));
                    };
                    if (block == 0) take(rec0);
                    else if (block == 1) take(rec1);
                    else if (block == 2) take(rec2);
                    else take(rec3);
                    tile_index = 64u * block + uint32_t(src);
                }
            }
        }
        const uint32_t count = run;
        if (WIDE) {
            // Two neighbouring tiles of an expert are one workgroup's work where the second continues the first's pairs (as
            // grouping leaves them; a caller's table may leave tiles out): the first of them takes both. A tile is a first one
            // where an even number of tiles ahead of it, each continuing the one before, run into it. The workgroup's place is
            // among the first ones of its XCD's run, so that the workgroups without a tile are the last ones. Where every tile had
            // its workgroups and those of the second ones left at once, the compute units did not fill evenly: 32 experts of
            // 2,880 x 2,880, 2,048 tokens 500 -> 483 us, 700 tokens 224 -> 217 (with the two tiles' workgroups in turn 680 and 318).
            // Within each 64 records the experts of one tile go last: the workgroups that start late are then the short ones (uneven
            // experts, both products, in the table's order against this: 64 of 2,048 x 512, 8-bit, 2,000 tokens 164 -> 160 us, 32 of
            // 2,880 x 2,880, 8-bit, 1,000 tokens 423 -> 398, 48 of 2,816 x 1,408, 4-bit, 1,500 tokens 277 -> 271).
            // What is left over of a longer expert stays behind that expert's other tiles, whose codes the L2 then has. Left-overs
            // last as well, against this: 256 even experts of 2,304 x 1,024, 8-bit, 4,000 tokens 766, 713 us; 256 of 2,048 x 512,
            // 4-bit, 4,096 tokens, whole pass 491, 475; 128 of 3,072 x 1,024, 8-bit, 2,000 tokens 514, 492; 32 of 3,072 x 2,048, 8-bit,
            // 700 tokens 369, 351; but 32 of 2,880 x 2,880, 4-bit, 2,048 tokens 478, 490 and 48 of 2,816 x 1,408, 4-bit 263, 279:
            // the short ones fill the end there. Over 29 shapes the two come to the same; the larger losses are last's.
            auto continues = [&](const uint4 &rec, const uint4 &before) {
                return rec.w == before.w && rec.x == before.x && before.z == kRowTile && rec.y == before.y + kRowTile;
            };
            auto record = [&](uint32_t at) { return at < tile_total ? table[at] : zero4(); };
            uint4 rec = record(first + lane), next = record(first + lane + 1u);
            // the tiles that run into the run's first one: lane l reads record at - l, the one before it is lane l + 1's
            uint32_t ahead = 0;
            for (uint32_t at = first;; at -= 63u) {
                const uint4 back = lane <= at ? record(at - lane) : zero4();
                const uint4 before = make_uint4(__shfl_down(back.x, 1), __shfl_down(back.y, 1), __shfl_down(back.z, 1), __shfl_down(back.w, 1));
                const uint64_t links = __ballot(lane < min(at, 63u) && continues(back, before));
                const uint32_t run_in = uint32_t(__ffsll((long long)~links)) - 1u;
                ahead += run_in;
                if (run_in < 63u) break;
            }
            bool found = false;
            uint32_t rank = place;
            for (uint32_t at = first; at < first + run && !found; at += 64u) {
                const bool goes_on = next.z != 0u && continues(next, rec);
                const uint64_t links = __ballot(goes_on) << 1;  // bit l: record at + l continues the one before it
                const uint64_t breaks = ~links & ((2ull << lane) - 1ull);  // (bit 0 always: `ahead` is what runs into it)
                const uint32_t from = 63u - uint32_t(__clzll((long long)breaks)), mine_ahead = lane - from + (from == 0u ? ahead : 0u);
                const bool is_first = at + lane < first + run && (mine_ahead & 1u) == 0u;
                const uint32_t rows = rec.z + (goes_on ? next.z : 0u);
                const bool is_heavy = rows > kRowTile || mine_ahead != 0u;
                const uint64_t heavy = __ballot(is_first && is_heavy), light = __ballot(is_first && !is_heavy);
                const uint32_t heavies = uint32_t(__popcll(heavy)), firsts = heavies + uint32_t(__popcll(light));
                if (rank < firsts) {
                    const uint64_t set = rank < heavies ? heavy : light;
                    const uint32_t want = rank < heavies ? rank : rank - heavies;
                    const bool me = ((set >> lane) & 1ull) != 0ull && uint32_t(__popcll(set & ((1ull << lane) - 1ull))) == want;
                    const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(me)) - 1);
                    tile.cell = uint32_t(__builtin_amdgcn_readlane(int(rec.x), src));
                    tile.pair_start = uint32_t(__builtin_amdgcn_readlane(int(rec.y), src));
                    tile.rows = uint32_t(__builtin_amdgcn_readlane(int(rows), src));
                    tile.expert = uint32_t(__builtin_amdgcn_readlane(int(rec.w), src));
                    tile_index = at + uint32_t(src);
                    found = true;
                }
                rank -= firsts;
                // what runs into the next 64's first record
                const uint32_t last_ahead = uint32_t(__builtin_amdgcn_readlane(int(mine_ahead), 63));
                ahead = __builtin_amdgcn_readlane(int(goes_on), 63) ? last_ahead + 1u : 0u;
                if (!found && at + 64u < first + run) {
                    rec = record(at + 64u + lane);
                    next = record(at + 65u + lane);
                }
            }
            if (!found) return;
        } else if (chosen) {
        } else if (count <= 64u) {
            const uint4 rec = lane < count ? table[first + lane] : zero4();
            const uint64_t heavy = __ballot(lane < count && rec.z > 32u), light = __ballot(lane < count && rec.z <= 32u);
            const uint32_t heavies = uint32_t(__popcll(heavy));
            const uint64_t set = place < heavies ? heavy : light;
            const uint32_t want = place < heavies ? place : place - heavies;
            const bool mine = ((set >> lane) & 1ull) != 0ull && uint32_t(__popcll(set & ((1ull << lane) - 1ull))) == want;
            const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(mine)) - 1);
            tile.cell = uint32_t(__builtin_amdgcn_readlane(int(rec.x), src));
            tile.pair_start = uint32_t(__builtin_amdgcn_readlane(int(rec.y), src));
            tile.rows = uint32_t(__builtin_amdgcn_readlane(int(rec.z), src));
            tile.expert = uint32_t(__builtin_amdgcn_readlane(int(rec.w), src));
            tile_index = first + uint32_t(src);
        } else {
            tile = a.tiles[tile_index];
        }
        if (a.residency) {  // moe.metal:136-146: a hit names its cell, anything else is the sentinel
            const uint64_t word = a.residency[tile.expert];
            tile.cell = uint32_t(word >> 32) == SHRIKE_RESIDENCY_RESIDENT ? uint32_t(word) : kSentinel;
        }
        if (tile.cell == kSentinel || tile.rows == 0) return;
        if (tile.pair_start + tile.rows <= a.pair_lo || tile.pair_start >= a.pair_hi) return;
    }

    const uint32_t act_row = tile_index * kRowTile + skip;
    // Whether the tile asks for its codes past the caches: it is its expert's last, not full, and whole, and the next launch would
    // not find them in the memory-side cache either. The experts in use are counted by such tiles in the first 256 records, so
    // those of a multiple of 64 pairs and of later records are left out: never too many. An expert of more than 64 rows has other
    // tiles that ask for the same lines without the hint. That costs nothing that shows: with the hint for experts of one tile only,
    // 1,000 uneven tokens of 256 x 2,304 x 1,024 331 to 335 us in three runs, like this 331 to 333; 600 of 128 149 to 151, 149 to 151.
    bool once = false;
    if constexpr (S == FfnShape::kLines) {
        auto last_tiles = [&](const uint4 &rec, uint32_t at) { return uint32_t(__popcll(__ballot(lane + at < tile_total && rec.z < kRowTile))); };
        const uint32_t in_use = last_tiles(rec0, 0) + last_tiles(rec1, 64) + last_tiles(rec2, 128) + last_tiles(rec3, 192);
        const bool in_two = larger != 0u && ((larger >> tile_index) & 1u) != 0u;
        once = tile.rows < kRowTile && !in_two && past_the_cache(in_use, a.d, a.f, BITS);
    }
    if (WIDE && tile.rows > 96u) ffn_tile<BITS, MODE, DENSE, WIDE ? 4 : 2, META, S>(a, tile, act_row, col_block, lds, once);
    else if (WIDE && tile.rows > 64u) ffn_tile<BITS, MODE, DENSE, WIDE ? 3 : 2, META, S>(a, tile, act_row, col_block, lds, once);
    else if (tile.rows > 32u) ffn_tile<BITS, MODE, DENSE, 2, META, S>(a, tile, act_row, col_block, lds, once);
    else ffn_tile<BITS, MODE, DENSE, 1, META, S>(a, tile, act_row, col_block, lds, once);
}

// ---- few rows: the same products with k split over the waves.
//
// Where k_grouped_ffn would leave most of the chip idle (a short chunk, or the shared expert: 512 tokens of one expert are
// eight row tiles of four column blocks), a workgroup's walk over k is a chain of a microsecond for three groups, whatever
// its rows. Here a workgroup takes up to 32 rows against 64 weight rows (32 of the gate and 32 of the up product), a quarter
// of k a wave, and the four partial sums meet in LDS in the order of k at the end: an eighth of the columns and a quarter of
// the walk. The operands come through LDS as in ffn_tile, each wave's its own, so the loop has no barrier. The bias term
// needs no sums from elsewhere: a wave adds up its rows while it multiplies them, and four groups of them meet their biases in
// one MFMA (the lanes' two halves of a group are two of its k). Two workgroups a compute unit, two groups of operands in
// flight; deeper rings at one workgroup a compute unit were slower (20 against 16 us below): what bounds it is the start and
// the end of a piece, some 4 us, which a neighbour hides, not the loads between them.
// The shared expert of 2,048 x 512, 4-bit: 45 -> 13 us for 37 rows, 49 -> 16 for 512.
template <int BITS, int MODE, bool DENSE, int META>
__global__ __launch_bounds__(256, 2) void k_ffn_split(FfnArgs a) {
    warm_kernel_arguments(a);
    extern __shared__ __align__(16) uint8_t lds[];
    typedef SplitLds L;
    const uint32_t lane = threadIdx.x & 63u, wave = wave_index();
    const uint32_t col = lane & 31u, kb = lane >> 5;
    const uint32_t K = MODE == 0 ? a.d : a.f, N = MODE == 0 ? a.f : a.d, G = K / kGroup;
    constexpr uint32_t kColumns = MODE == 0 ? 32u : 64u;  // of the output
    constexpr uint32_t kGroupsPerB = BITS == 4 ? 2u : 1u;
    const uint32_t stages = (G + kGroupsPerB - 1u) / kGroupsPerB, row_bytes = K * BITS / 8u;
    // the wave's quarter of the stages
    const uint32_t st_lo = stages * wave / 4u, st_hi = stages * (wave + 1u) / 4u;
    const uint32_t g_lo = st_lo * kGroupsPerB, g_hi = min(st_hi * kGroupsPerB, G), groups = g_hi - g_lo;
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)lds)) + wave * L::kWave;
    const uint8_t *my_lds = lds + wave * L::kWave;
    // An XCD takes a contiguous eighth of the (tile, column block) pairs, its workgroups one after the other: tiles of an
    // expert share its codes there, the column blocks of a tile its rows.
    const uint32_t column_blocks = N / kColumns;
    const uint32_t total_items = (DENSE ? (a.dense_rows + 31u) / 32u : *a.tile_count) * column_blocks;
    const uint32_t xcd = blockIdx.x & 7u, run = total_items / 8u + (xcd < total_items % 8u ? 1u : 0u);
    const uint32_t run_first = xcd * (total_items / 8u) + min(xcd, total_items % 8u);
    for (uint32_t place = blockIdx.x >> 3; place < run; place += gridDim.x >> 3) {
        const uint32_t item = run_first + place;
        uint32_t tile_index, col_block;
        shrike_row_tile tile;
        if (DENSE) {  // the rows of a column block are neighbours
            const uint32_t row_tiles = total_items / column_blocks;
            col_block = item / row_tiles;
            tile_index = item % row_tiles;
            tile.cell = 0;
            tile.pair_start = tile_index * 32u;
            tile.rows = min(32u, a.dense_rows - tile.pair_start);
        } else {
            tile_index = item / column_blocks;
            col_block = item % column_blocks;
            tile = a.tiles[tile_index];
            if (a.residency) {  // moe.metal:136-146: a hit names its cell, anything else is the sentinel
                const uint64_t word = a.residency[tile.expert];
                tile.cell = uint32_t(word >> 32) == SHRIKE_RESIDENCY_RESIDENT ? uint32_t(word) : kSentinel;
            }
            if (tile.cell == kSentinel) continue;
            if (tile.pair_start + tile.rows <= a.pair_lo || tile.pair_start >= a.pair_hi) continue;
        }
        const uint32_t n0 = col_block * kColumns;
        const uint8_t *base = DENSE ? nullptr : cell_base_uniform(a.pool, tile.cell, a.stride);
        const uint8_t *w_base[2];
        const uint16_t *s_base[2], *b_base[2];
        uint32_t n_first[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            n_first[nt] = n0 + (MODE == 0 ? 0u : 32u * uint32_t(nt));
            if (DENSE) {
                const int p = MODE == 0 ? nt : 2;
                w_base[nt] = a.dense_w[p]; s_base[nt] = a.dense_s[p]; b_base[nt] = a.dense_b[p];
            } else {
                w_base[nt] = base + (MODE != 0 ? a.off.down_w_off : nt ? a.off.up_w_off : a.off.gate_w_off);
                s_base[nt] = reinterpret_cast<const uint16_t *>(base + (MODE != 0 ? a.off.down_s_off : nt ? a.off.up_s_off : a.off.gate_s_off));
                b_base[nt] = reinterpret_cast<const uint16_t *>(base + (MODE != 0 ? a.off.down_b_off : nt ? a.off.up_b_off : a.off.gate_b_off));
            }
        }
        uint32_t b_off[4];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j)
            b_off[j] = (n_first[j >> 1] + 16u * (j & 1u) + (lane >> 2)) * row_bytes + ((lane & 3u) ^ ((lane >> 3) & 3u)) * 16u;
        const uint32_t half_back = (((lane & 3u) ^ ((lane >> 3) & 3u)) & 2u) * 16u;
        auto load_b = [&](uint32_t slot, uint32_t stage) {
            const uint32_t back = BITS == 4 && 2u * stage + 1u >= G ? half_back : 0u;
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) lds_load16(lds0 + L::kB + slot * kUnitB + j * 1024u, w_base[j >> 1] + size_t(stage) * 64u, b_off[j] - back);
        };
        // scales and biases: a window of three words a row, as in ffn_tile
        struct Run { const uint8_t *src; uint32_t mine, mine_last, at[2], last[2]; };
        auto make_run = [&](const uint16_t *const (&b)[2]) {
            Run r;
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                const uint32_t skew = uint32_t(reinterpret_cast<uintptr_t>(b[nt]) & 3u);
                r.at[nt] = skew + ((n_first[nt] + col) * G + g_lo) * 2u;
                r.last[nt] = ((skew + N * G * 2u + 3u) & ~3u) - 12u;
            }
            const uint8_t *p = reinterpret_cast<const uint8_t *>(kb ? b[1] : b[0]);
            r.src = p - (reinterpret_cast<uintptr_t>(p) & 3u);
            r.mine = kb ? r.at[1] : r.at[0];
            r.mine_last = kb ? r.last[1] : r.last[0];
            return r;
        };
        const Run rs = make_run(s_base), rb = make_run(b_base);
        auto load_s = [&](uint32_t c) {
            lds_load12(lds0 + L::kS, rs.src + min((rs.mine & ~3u) + 8u * c, rs.mine_last));
            lds_load12(lds0 + L::kBias, rb.src + min((rb.mine & ~3u) + 8u * c, rb.mine_last));
        };
        auto read_run = [&](const Run &r, uint32_t area, uint32_t i0, uint32_t (&v)[2][4]) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                const int into = max(int(r.at[nt] & 3u), int(r.at[nt] + i0 * 2u) - int(r.last[nt]));
                const uint8_t *p = my_lds + area + (uint32_t(nt) * 32u + col) * 16u + uint32_t(into);
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i) v[nt][i] = *reinterpret_cast<const uint16_t *>(p + min(i, groups - 1u - i0) * 2u);
            }
        };

        for (uint32_t skip = 0; skip < tile.rows; skip += 32u) {  // (dense: once)
            const uint32_t rows = min(32u, tile.rows - skip), first = tile.pair_start + skip;
            const uint32_t act_row = DENSE ? first : tile_index * kRowTile + skip;
            f32x16 total[2];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int i = 0; i < 16; ++i) total[nt][i] = 0.0f;
            // (rows past the last eight that hold one are not loaded: what the LDS holds there is multiplied into rows that
            // nobody reads)
            auto walk = [&](auto loads_a) {
                constexpr uint32_t kLoadsA = decltype(loads_a)::value;
                const uint8_t *a_src[kLoadsA];
#pragma unroll
                for (uint32_t j = 0; j < kLoadsA; ++j) {
                    const uint32_t r = min(8u * j + (lane >> 3), rows - 1u);
                    const uint16_t *row = MODE != 0 ? a.act + size_t(act_row + r) * a.f
                                                    : a.hidden + size_t(DENSE ? first + r : a.pairs[first + r].token) * a.hidden_stride;
                    a_src[j] = reinterpret_cast<const uint8_t *>(row + g_lo * kGroup) + (((lane & 7u) ^ (lane >> 3)) * 16u);
                }
                auto load_a = [&](uint32_t slot, uint32_t i) {
#pragma unroll
                    for (uint32_t j = 0; j < kLoadsA; ++j) lds_load16(lds0 + slot * L::kUnitA + j * 1024u, a_src[j] + size_t(i) * 128u);
                };
                if (groups != 0u) {
                    load_s(0);
                    load_b(0, st_lo);
                    load_a(0, 0);
                }
                uint32_t run_s[2][4], run_b[2][4];
                Frag sums;  // of the chunk's groups: the lane's row over its half of each group's k, hi and lo
                auto step = [&](uint32_t i, auto par) {
                    constexpr uint32_t P = decltype(par)::value;
                    const uint32_t b_place = BITS == 8 ? P : (i >> 1) & 1u;
                    if (BITS == 4 && P == 1u && i + 1u < groups) wait_loads<4>();  // (the next stage's codes may still be on their way)
                    else wait_loads<0>();
                    if (i + 1u < groups) {
                        load_a(P ^ 1u, i + 1u);
                        if (BITS == 8) load_b(b_place ^ 1u, st_lo + i + 1u);
                    }
                    if (BITS == 4 && P == 0u && i + 2u < groups) load_b(b_place ^ 1u, st_lo + (i >> 1) + 1u);
                    const uint32_t in_chunk = i & 3u;
                    if (in_chunk == 0u) {
                        read_run(rs, L::kS, i, run_s);
                        read_run(rb, L::kBias, i, run_b);
                        sums.v = zero4();
                    }
                    if (in_chunk == 1u && i + 3u < groups) load_s((i >> 2) + 1u);
                    const uint8_t *a_rows = my_lds + P * L::kUnitA + col * 128u;
                    Frag af[4];
#pragma unroll
                    for (uint32_t s = 0; s < 4u; ++s) af[s].v = *reinterpret_cast<const uint4 *>(a_rows + (((kb * 4u + s) ^ (col & 7u)) * 16u));
                    float sum = 0.0f;
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt) {
                        const uint8_t *b_rows = my_lds + L::kB + b_place * kUnitB + uint32_t(nt) * 2048u + col * 64u;
                        uint4 codes[BITS / 4];
#pragma unroll
                        for (uint32_t j = 0; j < BITS / 4; ++j)
                            codes[j] = *reinterpret_cast<const uint4 *>(b_rows + (((BITS == 4 ? P * 2u + kb : kb * 2u + j) ^ ((col >> 1) & 3u)) * 16u));
                        half8 bf[4];
                        if (BITS == 4) {
                            bf[0] = codes4(codes[0].x); bf[1] = codes4(codes[0].y); bf[2] = codes4(codes[0].z); bf[3] = codes4(codes[0].w);
                        } else {
                            const uint4 lo = codes[0], hi = codes[BITS / 4 - 1];
                            bf[0] = codes8(lo.x, lo.y); bf[1] = codes8(lo.z, lo.w); bf[2] = codes8(hi.x, hi.y); bf[3] = codes8(hi.z, hi.w);
                        }
                        f32x16 p = {0};
#pragma unroll
                        for (int s = 0; s < 4; ++s) p = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[s].h, bf[s], p, 0, 0, 0);
                        if (nt == 0) {
#pragma unroll
                            for (int s = 0; s < 4; ++s)
#pragma unroll
                                for (int w = 0; w < 4; ++w) sum = dot2_ones(af[s].u[w], sum);
                        }
                        const float scale = meta_f32(uint16_t(run_s[nt][0]), uint32_t(META)) * kTwo24;
                        run_s[nt][0] = run_s[nt][1]; run_s[nt][1] = run_s[nt][2]; run_s[nt][2] = run_s[nt][3];
#pragma unroll
                        for (int j = 0; j < 16; ++j) total[nt][j] = fmaf(scale, p[j], total[nt][j]);
                    }
                    const uint32_t hi_lo = split_hi_lo(sum);
                    if (in_chunk == 0u) sums.u[0] = hi_lo;
                    else if (in_chunk == 1u) sums.u[1] = hi_lo;
                    else if (in_chunk == 2u) sums.u[2] = hi_lo;
                    else sums.u[3] = hi_lo;
                    if (in_chunk == 3u || i + 1u == groups) {  // the bias term of a chunk: one MFMA
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt) {
                            Frag f;
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const uint16_t bits = META == SHRIKE_META_BF16 ? f32_to_f16(bf16_to_f32(uint16_t(run_b[nt][j]))) : uint16_t(run_b[nt][j]);
                                f.u[j] = uint32_t(bits) * (uint32_t(j) <= in_chunk ? 0x00010001u : 0u);  // (past the last group a copy: zero times it may be no zero)
                            }
                            total[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums.h, f.h, total[nt], 0, 0, 0);
                        }
                    }
                };
                for (uint32_t i = 0; i + 1u < groups; i += 2u) {
                    step(i, std::integral_constant<uint32_t, 0>{});
                    step(i + 1u, std::integral_constant<uint32_t, 1>{});
                }
                if (groups & 1u) step(groups - 1u, std::integral_constant<uint32_t, 0>{});
            };
            if (rows <= 8u) walk(std::integral_constant<uint32_t, 1>{});
            else if (rows <= 16u) walk(std::integral_constant<uint32_t, 2>{});
            else walk(std::integral_constant<uint32_t, 4>{});
            // ---- the quarters meet: eight threads a row
            __syncthreads();
            float (*s_part)[32][64] = reinterpret_cast<float (*)[32][64]>(lds);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int i = 0; i < 16; ++i) s_part[wave][8u * (i / 4) + 4u * kb + (i % 4)][32u * nt + col] = total[nt][i];
            __syncthreads();
            const uint32_t r = threadIdx.x >> 3, e = threadIdx.x & 7u;
            float v[8];  // MODE 0: four columns of the gate, then of the up product; MODE 1: eight columns
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t c = MODE == 0 ? 32u * h + 4u * e : 8u * e + 4u * h;
                float4 t = *reinterpret_cast<const float4 *>(&s_part[0][r][c]);
#pragma unroll
                for (int q = 1; q < 4; ++q) {
                    const float4 u = *reinterpret_cast<const float4 *>(&s_part[q][r][c]);
                    t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w;
                }
                v[4 * h] = t.x; v[4 * h + 1] = t.y; v[4 * h + 2] = t.z; v[4 * h + 3] = t.w;
            }
            if (r < rows) {
                if (MODE == 0) {
                    const uint32_t n = n0 + 4u * e;
                    uint32_t y[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float g = v[j], u = v[4 + j];
                        if (!DENSE && a.ebias) {  // moe.metal:261-269
                            g += bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.gate_ab_off)[n + j]);
                            u += bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.up_ab_off)[n + j]);
                        }
                        if (DENSE && a.round_gate_up) {
                            g = f16_to_f32(f32_to_f16(g));
                            u = f16_to_f32(f32_to_f16(u));
                        }
                        y[j] = f32_to_f16(glu_rt_fast(g, u, a.act_kind));
                    }
                    *reinterpret_cast<uint2 *>(a.act + size_t(act_row + r) * a.f + n) = make_uint2(y[0] | y[1] << 16, y[2] | y[3] << 16);
                } else if (DENSE || (first + r >= a.pair_lo && first + r < a.pair_hi)) {
                    const uint32_t n = n0 + 8u * e;
                    float gate_mul = 1.0f;
                    if (DENSE && a.scalar_gate) gate_mul = 1.0f + expf(-f16_to_f32(a.scalar_gate[first + r]));  // one gate a token row (moe.metal:1195-1207)
                    uint16_t *to;
                    if (DENSE) {
                        to = a.partials + size_t(first + r) * a.d;
                    } else {
                        const shrike_token_expert_pair p = a.pairs[first + r];
                        to = a.partials + (size_t(p.token) * a.top_k + p.rank) * a.d;
                    }
                    uint32_t y[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        float o = v[j];
                        if (!DENSE && a.ebias) o += bf16_to_f32(reinterpret_cast<const uint16_t *>(base + a.off.down_ab_off)[n + j]);
                        y[j] = f32_to_f16(o);
                        if (DENSE && a.scalar_gate) y[j] = f32_to_f16(f16_to_f32(uint16_t(y[j])) / gate_mul);
                    }
                    *reinterpret_cast<uint4 *>(to + n) = make_uint4(y[0] | y[1] << 16, y[2] | y[3] << 16, y[4] | y[5] << 16, y[6] | y[7] << 16);
                }
            }
            __syncthreads();  // the partial sums have been read: the next rows' operands may land
        }
    }
}

int launch_row_group_sums(const uint16_t *src, size_t stride, uint32_t rows, uint32_t n, uint32_t *out,
                          const uint32_t *row_limit_tiles, hipStream_t s);

static uint32_t compute_units() {
    int device = 0, units = 0;
    if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return 0;
    return uint32_t(units);
}

template <int BITS, bool DENSE, int META, FfnShape S>
static int launch_ffn_shape(FfnArgs a, uint32_t max_tiles, hipStream_t s) {
    a.resident_workgroups = Lds<S, BITS>::kResident * compute_units();
    const dim3 block(256);
    const uint32_t grid_tiles = (max_tiles + 7u) & ~7u;  // whole runs for the kernel's XCD mapping
    hipLaunchKernelGGL((k_grouped_ffn<BITS, 0, DENSE, META, S>), dim3(grid_tiles, (a.f + 127u) / 128u), block, 0, s, a);
    SHRIKE_HIP(hipGetLastError());
    // (the activations' group sums were written by the gate/up launch itself)
    hipLaunchKernelGGL((k_grouped_ffn<BITS, 1, DENSE, META, S>), dim3(grid_tiles, (a.d + 255u) / 256u), block, 0, s, a);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}
template <int BITS, bool DENSE, int META>
static int launch_ffn_split(const FfnArgs &a, uint32_t max_tiles, hipStream_t s) {
    const uint32_t tiles = DENSE ? (a.dense_rows + 31u) / 32u : max_tiles;
    auto grid = [&](uint32_t column_blocks) { return dim3((uint32_t(min(uint64_t(tiles) * column_blocks, uint64_t(2u * compute_units()))) + 7u) & ~7u); };
    hipLaunchKernelGGL((k_ffn_split<BITS, 0, DENSE, META>), grid(a.f / 32u), dim3(256), SplitLds::kBytes, s, a);
    SHRIKE_HIP(hipGetLastError());
    hipLaunchKernelGGL((k_ffn_split<BITS, 1, DENSE, META>), grid(a.d / 64u), dim3(256), SplitLds::kBytes, s, a);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

template <int BITS, bool DENSE, int META>
static int launch_ffn_meta(const FfnArgs &a, uint32_t max_tiles, FfnShape shape, hipStream_t s) {
    if (shape == FfnShape::kSplit) return launch_ffn_split<BITS, DENSE, META>(a, max_tiles, s);
    if constexpr (!DENSE)
        if (shape == FfnShape::kWide) return launch_ffn_shape<BITS, DENSE, META, FfnShape::kWide>(a, max_tiles, s);
    if constexpr (!DENSE && BITS == 8)
        if (shape == FfnShape::kLines) return launch_ffn_shape<BITS, DENSE, META, FfnShape::kLines>(a, max_tiles, s);
    if constexpr (!DENSE && BITS == 4)
        if (shape == FfnShape::kTile) return launch_ffn_shape<BITS, DENSE, META, FfnShape::kTile>(a, max_tiles, s);
    return launch_ffn_shape<BITS, DENSE, META, FfnShape::kDeep>(a, max_tiles, s);
}
template <int BITS, bool DENSE>
static int launch_ffn(const FfnArgs &a, uint32_t max_tiles, FfnShape shape, hipStream_t s) {
    return a.meta == SHRIKE_META_F16 ? launch_ffn_meta<BITS, DENSE, SHRIKE_META_F16>(a, max_tiles, shape, s)
                                     : launch_ffn_meta<BITS, DENSE, SHRIKE_META_BF16>(a, max_tiles, shape, s);
}

struct Workspace {
    size_t hidden_sums, act, act_sums, total;
};
static Workspace workspace_layout(uint32_t query_count, uint32_t max_tiles, uint32_t d, uint32_t f) {
    auto round = [](size_t v) { return (v + 255u) & ~size_t(255); };
    Workspace w;
    w.hidden_sums = 0;
    w.act = round(size_t(query_count) * (d / kGroup) * 4u);
    w.act_sums = w.act + round(size_t(max_tiles) * kRowTile * f * 2u);
    w.total = w.act_sums + round(size_t(max_tiles) * kRowTile * (f / kGroup) * 4u);
    return w;
}

}  // namespace shrike

using namespace shrike;

extern "C" {
size_t shrike_hip_prefill_ffn_workspace_bytes(uint32_t query_count, uint32_t max_row_tiles, uint32_t d, uint32_t f) {
    return workspace_layout(query_count, max_row_tiles, d, f).total;
}

static int grouped_ffn(shrike_hip_moe *moe, void *stream, const shrike_pool_bases *pool, uint64_t pool_slot_stride,
                       const shrike_expert_offsets *offsets, const shrike_hip_grouped_routes *routes, uint32_t max_row_tiles,
                       const uint64_t *d_residency, uint32_t pair_lo, uint32_t pair_hi, const void *d_hidden,
                       uint32_t hidden_stride_elements, void *d_route_partials, void *d_workspace, size_t workspace_bytes,
                       uint32_t query_count, uint32_t d, uint32_t f, uint32_t top_k, bool presummed = false) {
    SHRIKE_REQUIRE(moe && pool && offsets && routes, "grouped FFN: NULL argument");
    SHRIKE_REQUIRE(d == moe->desc.d && f == moe->desc.f, "grouped FFN: shape %ux%u differs from the handle's %ux%u", d, f, moe->desc.d, moe->desc.f);
    SHRIKE_REQUIRE(d % kGroup == 0 && f % kGroup == 0 && d > 0 && f > 0, "D and F must be positive multiples of 64");
    SHRIKE_REQUIRE(top_k > 0, "topK must be positive");
    SHRIKE_REQUIRE(hidden_stride_elements >= d && hidden_stride_elements % 8u == 0, "hidden stride is too small or leaves rows unaligned");
    SHRIKE_REQUIRE(routes->sorted_pairs && routes->row_tiles && routes->row_tile_count, "grouped FFN: routes are not bound");
    SHRIKE_REQUIRE(d_hidden && d_route_partials && d_workspace, "grouped FFN: NULL buffer");
    SHRIKE_REQUIRE(reinterpret_cast<uintptr_t>(d_workspace) % 256u == 0, "grouped FFN: workspace must be 256-byte aligned");
    SHRIKE_REQUIRE(pool->cells_per_chunk > 0 && pool_slot_stride % 16u == 0, "grouped FFN: bad pool geometry");
    if (int rc = check_offsets(offsets, d, f, moe->desc.routed_weight_bits)) return rc;
    if (max_row_tiles == 0 || query_count == 0 || pair_lo >= pair_hi) return 0;
    const Workspace w = workspace_layout(query_count, max_row_tiles, d, f);
    SHRIKE_REQUIRE(workspace_bytes >= w.total, "grouped FFN: workspace of %zu bytes, %zu needed", workspace_bytes, w.total);
    uint8_t *ws = static_cast<uint8_t *>(d_workspace);
    FfnArgs a = {};
    fill_pool(a.pool, pool);
    a.stride = pool_slot_stride;
    a.off = *offsets;
    a.tiles = routes->row_tiles;
    a.tile_count = routes->row_tile_count;
    a.table_room = readable_records(max_row_tiles, uint64_t(query_count) * top_k, moe->desc.num_experts);
    a.residency = d_residency;
    a.pair_lo = pair_lo;
    a.pair_hi = pair_hi;
    a.pairs = static_cast<const shrike_token_expert_pair *>(routes->sorted_pairs);
    a.hidden = static_cast<const uint16_t *>(d_hidden);
    a.hidden_stride = hidden_stride_elements;
    a.hidden_sums = reinterpret_cast<uint32_t *>(ws + w.hidden_sums);
    a.act = reinterpret_cast<uint16_t *>(ws + w.act);
    a.act_sums = reinterpret_cast<uint32_t *>(ws + w.act_sums);
    a.partials = static_cast<uint16_t *>(d_route_partials);
    a.d = d; a.f = f; a.top_k = top_k;
    a.meta = moe->desc.meta_dtype;
    a.act_kind = moe->desc.activation;
    a.ebias = moe->desc.expert_additive_biases;
    hipStream_t s = as_stream(stream);
    if (!presummed)
        if (int rc = launch_row_group_sums(a.hidden, hidden_stride_elements, query_count, d, const_cast<uint32_t *>(a.hidden_sums), nullptr, s)) return rc;
    FfnShape shape = routed_shape(uint64_t(query_count) * top_k, moe->desc.num_experts, d, f, moe->desc.routed_weight_bits);
    uint64_t align = pool_slot_stride | offsets->gate_w_off | offsets->up_w_off | offsets->down_w_off | d | f;  // (a row of 8-bit codes is d or f bytes)
    for (const void *base : pool->base) align |= reinterpret_cast<uintptr_t>(base);
    shape = lines_shape(shape, uint64_t(query_count) * top_k, moe->desc.num_experts, d, f, moe->desc.routed_weight_bits, align);
    if (shape != FfnShape::kSplit && uint64_t(query_count) * hidden_stride_elements * 2u > 0xffffffffull) shape = FfnShape::kDeep;  // (the others' rows are 32-bit offsets)
    return moe->desc.routed_weight_bits == 8 ? launch_ffn<8, false>(a, max_row_tiles, shape, s) : launch_ffn<4, false>(a, max_row_tiles, shape, s);
}

int shrike_hip_prefill_grouped_ffn(shrike_hip_moe *moe, void *stream, const shrike_pool_bases *pool,
                                   uint64_t pool_slot_stride, const shrike_expert_offsets *offsets,
                                   const shrike_hip_grouped_routes *routes, uint32_t max_row_tiles, const void *d_hidden,
                                   uint32_t hidden_stride_elements, void *d_route_partials, void *d_workspace,
                                   size_t workspace_bytes, uint32_t query_count, uint32_t d, uint32_t f, uint32_t top_k) {
    return grouped_ffn(moe, stream, pool, pool_slot_stride, offsets, routes, max_row_tiles, nullptr, 0u, 0xffffffffu, d_hidden,
                       hidden_stride_elements, d_route_partials, d_workspace, workspace_bytes, query_count, d, f, top_k);
}

int shrike_hip_prefill_grouped_ffn_presummed(shrike_hip_moe *moe, void *stream, const shrike_pool_bases *pool,
                                             uint64_t pool_slot_stride, const shrike_expert_offsets *offsets,
                                             const shrike_hip_grouped_routes *routes, uint32_t max_row_tiles,
                                             const void *d_hidden, uint32_t hidden_stride_elements, void *d_route_partials,
                                             void *d_workspace, size_t workspace_bytes, uint32_t query_count, uint32_t d,
                                             uint32_t f, uint32_t top_k) {
    return grouped_ffn(moe, stream, pool, pool_slot_stride, offsets, routes, max_row_tiles, nullptr, 0u, 0xffffffffu, d_hidden,
                       hidden_stride_elements, d_route_partials, d_workspace, workspace_bytes, query_count, d, f, top_k, true);
}

int shrike_hip_prefill_streamed_batched(shrike_hip_moe *moe, void *stream, const shrike_pool_bases *pool,
                                        uint64_t pool_slot_stride, const shrike_expert_offsets *offsets,
                                        const shrike_hip_grouped_routes *routes, uint32_t max_row_tiles,
                                        const uint64_t *d_residency, uint32_t pair_start, uint32_t pair_count,
                                        uint32_t pair_microbatch_rows, const void *d_hidden, uint32_t hidden_stride_elements,
                                        void *d_route_partials, void *d_workspace, size_t workspace_bytes,
                                        uint32_t query_count, uint32_t d, uint32_t f, uint32_t top_k,
                                        uint32_t *out_microbatches) {
    if (out_microbatches) *out_microbatches = 0;
    // PrefillGroupedRoutedMoE.swift:861-863: nothing to do is not an error
    if (pair_count == 0 || pair_microbatch_rows == 0) return 0;
    SHRIKE_REQUIRE(uint64_t(pair_start) + pair_count <= uint64_t(query_count) * top_k, "streamed batch: pairs %u..%llu leave the chunk's %llu",
                   pair_start, (unsigned long long)pair_start + pair_count, (unsigned long long)query_count * top_k);
    if (int rc = grouped_ffn(moe, stream, pool, pool_slot_stride, offsets, routes, max_row_tiles, d_residency, pair_start,
                             pair_start + pair_count, d_hidden, hidden_stride_elements, d_route_partials, d_workspace,
                             workspace_bytes, query_count, d, f, top_k))
        return rc;
    if (out_microbatches) *out_microbatches = (pair_count + pair_microbatch_rows - 1u) / pair_microbatch_rows;
    return 0;
}

size_t shrike_hip_prefill_shared_expert_workspace_bytes(uint32_t query_count, uint32_t d, uint32_t f_shared) {
    return workspace_layout(query_count, (query_count + kRowTile - 1u) / kRowTile, d, f_shared).total;
}

int shrike_hip_prefill_shared_expert(shrike_hip_moe *moe, void *stream, const shrike_projection *gate,
                                     const shrike_projection *up, const shrike_projection *down, uint32_t bits,
                                     const void *d_hidden, uint32_t hidden_stride_elements, void *d_h1, const void *d_scalar_gate,
                                     void *d_workspace, size_t workspace_bytes, uint32_t query_count, uint32_t d,
                                     uint32_t f_shared) {
    SHRIKE_REQUIRE(moe != nullptr, "moe handle is NULL");
    if (int rc = check_shared(gate, up, down, bits, d, f_shared)) return rc;
    SHRIKE_REQUIRE(hidden_stride_elements >= d && hidden_stride_elements % 8u == 0, "hidden stride is too small or leaves rows unaligned");
    SHRIKE_REQUIRE(d_hidden && d_h1 && d_workspace, "shared expert: NULL buffer");
    SHRIKE_REQUIRE(reinterpret_cast<uintptr_t>(d_workspace) % 256u == 0, "shared expert: workspace must be 256-byte aligned");
    if (query_count == 0) return 0;
    const uint32_t tiles = (query_count + kRowTile - 1u) / kRowTile;
    const Workspace w = workspace_layout(query_count, tiles, d, f_shared);
    SHRIKE_REQUIRE(workspace_bytes >= w.total, "shared expert: workspace of %zu bytes, %zu needed", workspace_bytes, w.total);
    uint8_t *ws = static_cast<uint8_t *>(d_workspace);
    FfnArgs a = {};
    a.hidden = static_cast<const uint16_t *>(d_hidden);
    a.hidden_stride = hidden_stride_elements;
    a.hidden_sums = reinterpret_cast<uint32_t *>(ws + w.hidden_sums);
    a.act = reinterpret_cast<uint16_t *>(ws + w.act);
    a.act_sums = reinterpret_cast<uint32_t *>(ws + w.act_sums);
    a.partials = static_cast<uint16_t *>(d_h1);
    a.d = d; a.f = f_shared; a.top_k = 1;
    a.meta = moe->desc.meta_dtype;
    a.act_kind = moe->desc.activation;
    const shrike_projection *proj[3] = {gate, up, down};
    for (int i = 0; i < 3; ++i) {
        a.dense_w[i] = static_cast<const uint8_t *>(proj[i]->weights);
        a.dense_s[i] = static_cast<const uint16_t *>(proj[i]->scales);
        a.dense_b[i] = static_cast<const uint16_t *>(proj[i]->biases);
    }
    a.dense_rows = query_count;
    a.round_gate_up = 1;
    a.scalar_gate = static_cast<const uint16_t *>(d_scalar_gate);
    hipStream_t s = as_stream(stream);
    const FfnShape shape = dense_shape(query_count, f_shared);
    if (shape != FfnShape::kSplit)
        if (int rc = launch_row_group_sums(a.hidden, hidden_stride_elements, query_count, d, const_cast<uint32_t *>(a.hidden_sums), nullptr, s)) return rc;
    return bits == 8 ? launch_ffn<8, true>(a, tiles, shape, s) : launch_ffn<4, true>(a, tiles, shape, s);
}

}  // extern "C"
