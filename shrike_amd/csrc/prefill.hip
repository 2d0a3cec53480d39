// The prefill side of the routed path for gfx950, except the grouped FFN: the router for a
// block of tokens, the token->expert grouping as a stable counting sort, the per-row group
// sums the grouped FFN folds the affine biases with, the token-major reduce and the
// residual add.
#include "prefill_common.h"
#include <type_traits>
#include "router_row.h"
#include "router_rules.h"

#include "../../include/shrike_host.h"

namespace shrike {

// ---- router logits of a block of tokens (prefill.metal:369-439)
//
// x * effective_scale is the same for every expert: a workgroup forms the products (router_row's, moe.metal:357-358) once
// per token while staging the row in LDS, keeps its experts' rows in registers and walks a block of tokens, TPS of them a
// step, the next step's rows in flight while one is multiplied. The additions are router_row's, in router_row's order
// (lane l: chunks l, l + 64, ..., xor butterfly), so the logits are the decode router's bits.
//
// A wave keeps ROWS expert rows, MAXC 16-byte chunks a lane and row, as packed fp16: the fp16 rows as they are, the codes
// of an affine row widened once (every code is exact in fp16). A multiply-add that takes its fp16 factor as it is
// (v_fma_mix_f32) then widens it for nothing, and a row costs half the registers. An affine row's second operand, the
// chunk's sum of x, does not depend on the row either: it is formed while staging, in router_row's order.
//
// Bound by the vector unit: one multiply-add a code and token (55 us of them for 4,096 tokens of 2,048 against 256 rows).
// Router launches (logits and select), before and after the affine rows went this way and the butterfly left LDS: 8-bit
// rows, 1,000 tokens of 2,304 against 256: 195 -> 50 us; 4-bit rows, 512 of 2,048: 176 -> 24; fp16 rows, 1,000 of 2,304:
// 63 -> 36 (four rows a wave instead of two), 4,096 of 2,048: 94 -> 87.
// One stage of the split butterfly over LIVE sums (a power of two above 1) at lane distance 32 >> STAGE: the partner with
// the distance's bit set keeps the upper half of the sums and sends the lower, the other the reverse; each adds the
// partner's copy of what it keeps. LIVE / 2 sums are left in v[0 .. LIVE / 2). At distances 32 and 16 the exchange is one
// swap instruction a pair of sums (after it one register holds what the lane keeps and what its partner sent, the other
// the rest), at 8 a rotation within the row of sixteen lanes; none goes through LDS as a shuffle would.
template <uint32_t LIVE, uint32_t STAGE>
__device__ __forceinline__ void split_stage(float *v, uint32_t lane) {
    static_assert(STAGE <= 2u, "the split stages are those at distances 32, 16 and 8");
#pragma unroll
    for (uint32_t j = 0; j < LIVE / 2u; ++j) {
        const uint32_t a = __float_as_uint(v[j]), b = __float_as_uint(v[j + LIVE / 2u]);
        if constexpr (STAGE == 0u) {
            const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
            v[j] = __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
        } else if constexpr (STAGE == 1u) {
            const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
            v[j] = __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
        } else {
            const bool upper = (lane & 8u) != 0u;
            const float keep = __uint_as_float(upper ? b : a), send = __uint_as_float(upper ? a : b);
            v[j] = __fadd_rn(keep, dpp_f32<0x128>(send));  // row_ror:8
        }
    }
}

template <int RK, int MAXC, int ROWS, uint32_t TPS>
__global__ __launch_bounds__(256) void k_prefill_logits(RouterArgs a, uint32_t query_count, uint32_t stride, float *logits,
                                                        uint32_t tokens_a_group) {
    warm_kernel_arguments(a);
    constexpr int E = kRouterChunk<RK>, P = E / 4, W = E / 2;  // a chunk's elements, float4 of x, packed fp16 words
    // chunk c = lane + 64 i of a row is P float4: piece h sits at [(P i + h) * 64 + lane], so that a wave's read of one
    // piece is one contiguous kilobyte
    __shared__ float4 s_x[2][TPS][MAXC * P * 64];
    __shared__ float s_sum[RK ? 2 : 1][RK ? TPS : 1][RK ? MAXC * 64 : 1];
    const uint32_t lane = threadIdx.x & 63u, wave = wave_index();
    const uint32_t num_experts = a.sel.num_experts, d = a.d;
    const uint32_t e0 = (blockIdx.x * 4u + wave) * ROWS;
    const uint32_t chunks = d / E;
    uint32_t w[ROWS][MAXC][W];
    float sc[ROWS][MAXC], bi[ROWS][MAXC];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const uint32_t e = min(e0 + uint32_t(r), num_experts - 1u);  // past the last row: a copy, never stored
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const uint32_t c = lane + 64u * i, cc = c < chunks ? c : 0u;
            const uint4 v = *reinterpret_cast<const uint4 *>(static_cast<const uint8_t *>(a.weights) + (size_t(e) * chunks + cc) * 16u);
            const uint32_t vw[4] = {v.x, v.y, v.z, v.w};
            if (RK == 0) {
#pragma unroll
                for (int j = 0; j < 4; ++j) w[r][i][j] = vw[j];
            } else {
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    constexpr uint32_t mask = RK == 8 ? 0xffu : 0xfu;
                    const uint32_t pair = vw[j * RK / 16] >> ((2 * RK * j) % 32);
                    w[r][i][j] = as_u32(h2_t{_Float16(float(pair & mask)), _Float16(float((pair >> RK) & mask))});
                }
                sc[r][i] = meta_f32(a.scales[size_t(e) * (d / kGroup) + cc * E / kGroup], a.meta);
                bi[r][i] = meta_f32(a.biases[size_t(e) * (d / kGroup) + cc * E / kGroup], a.meta);
            }
        }
    }
    const uint32_t t0 = blockIdx.y * tokens_a_group;
    const uint32_t t1 = min(t0 + tokens_a_group, query_count);
    if (t0 >= t1) return;
    // a thread stages whole chunks of a token's row: fp16 x times bf16 effective scale, the exact fp32 product, P float4 a
    // chunk, and for an affine row the chunk's sum
    constexpr int kStage = (MAXC * 64 + 255) / 256, Q = E / 8;
    uint4 eff_c[kStage][Q];
#pragma unroll
    for (int j = 0; j < kStage; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q) eff_c[j][q] = reinterpret_cast<const uint4 *>(a.effective_scale)[min(threadIdx.x + 256u * j, chunks - 1u) * Q + q];
    auto stage_load = [&](uint4 (&st)[TPS][kStage][Q], uint32_t t) {
#pragma unroll
        for (uint32_t u = 0; u < TPS; ++u) {
            const uint4 *row = reinterpret_cast<const uint4 *>(a.hidden + size_t(min(t + u, t1 - 1u)) * stride);
#pragma unroll
            for (int j = 0; j < kStage; ++j)
#pragma unroll
                for (int q = 0; q < Q; ++q) st[u][j][q] = row[min(threadIdx.x + 256u * j, chunks - 1u) * Q + q];  // past the row: a copy, never stored
        }
    };
    auto stage_store = [&](const uint4 (&st)[TPS][kStage][Q], uint32_t buf) {
#pragma unroll
        for (uint32_t u = 0; u < TPS; ++u)
#pragma unroll
            for (int j = 0; j < kStage; ++j) {
                const uint32_t c = threadIdx.x + 256u * j;
                float sum = 0.0f;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const uint4 xv = st[u][j][q], ev = eff_c[j][q];
                    const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w}, ew[4] = {ev.x, ev.y, ev.z, ev.w};
                    float o[8];
#pragma unroll
                    for (int p = 0; p < 4; ++p) {  // moe.metal:357-358 (exact product)
                        o[2 * p] = __fmul_rn(f16_to_f32(uint16_t(xw[p])), bf16_to_f32(uint16_t(ew[p])));
                        o[2 * p + 1] = __fmul_rn(f16_to_f32(uint16_t(xw[p] >> 16)), bf16_to_f32(uint16_t(ew[p] >> 16)));
                    }
                    if (RK != 0)
#pragma unroll
                        for (int p = 0; p < 8; ++p) sum = __fadd_rn(sum, o[p]);
                    if (c < chunks) {
                        s_x[buf][u][(P * (c >> 6) + 2u * q) * 64u + (c & 63u)] = make_float4(o[0], o[1], o[2], o[3]);
                        s_x[buf][u][(P * (c >> 6) + 2u * q + 1u) * 64u + (c & 63u)] = make_float4(o[4], o[5], o[6], o[7]);
                    }
                }
                if (RK != 0 && c < chunks) s_sum[buf][u][c] = sum;
            }
    };
    auto step = [&](uint32_t buf, uint32_t t) {
        float acc[TPS][ROWS];
#pragma unroll
        for (uint32_t u = 0; u < TPS; ++u)
#pragma unroll
            for (int r = 0; r < ROWS; ++r) acc[u][r] = 0.0f;
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            if (lane + 64u * i < chunks) {
                // the widening belongs to the multiply-add: keep it from being hoisted out of the token loop. The row's own
                // registers are named as changed (they are not), so that nothing is copied for it.
#pragma unroll
                for (int r = 0; r < ROWS; ++r)
#pragma unroll
                    for (int j = 0; j < W; j += 4)
                        asm volatile("" : "+v"(w[r][i][j]), "+v"(w[r][i][j + 1]), "+v"(w[r][i][j + 2]), "+v"(w[r][i][j + 3]));
#pragma unroll
                for (uint32_t u = 0; u < TPS; ++u) {
                    float part[ROWS];
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) part[r] = RK == 0 ? acc[u][r] : 0.0f;
#pragma unroll
                    for (int h = 0; h < P; ++h) {
                        const float4 x4 = s_x[buf][u][(P * i + h) * 64 + lane];
                        const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                        for (int r = 0; r < ROWS; ++r)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                part[r] = fmaf(f16_to_f32(uint16_t(w[r][i][2 * h + j / 2] >> (16 * (j % 2)))), xv[j], part[r]);
                    }
                    if (RK == 0) {
#pragma unroll
                        for (int r = 0; r < ROWS; ++r) acc[u][r] = part[r];
                    } else {
                        const float sum = s_sum[buf][u][lane + 64u * i];
#pragma unroll
                        for (int r = 0; r < ROWS; ++r) acc[u][r] = fmaf(bi[r][i], sum, fmaf(sc[r][i], part[r], acc[u][r]));
                    }
                }
            }
        }
        // The butterfly of router_row (xor 32, 16, ..., 1) over the step's TPS * ROWS sums at once. While more than one
        // sum is left, a step's two partner lanes split them: each keeps half and adds the partner's copy of that half,
        // so a step costs half the exchanges of the one before; what a lane adds is what the plain butterfly adds in that
        // lane (the same two operands, and addition commutes), so every sum is router_row's bit for bit. Sum j ends in the
        // lanes whose upper bits spell j.
        constexpr uint32_t kSums = TPS * uint32_t(ROWS);
        static_assert(kSums == 4u || kSums == 8u, "the split butterfly takes 4 or 8 sums");
        float v[kSums];
#pragma unroll
        for (uint32_t u = 0; u < TPS; ++u)
#pragma unroll
            for (int r = 0; r < ROWS; ++r) v[u * ROWS + r] = acc[u][r];
        // (every index below is a constant: with the number of live sums in a variable the compiler kept v in private memory)
        split_stage<kSums, 0>(v, lane);
        split_stage<kSums / 2u, 1>(v, lane);
        if constexpr (kSums == 8u) split_stage<2u, 2>(v, lane);
        else v[0] = __fadd_rn(v[0], dpp_f32<0x128>(v[0]));  // row_ror:8
        v[0] = butterfly_from_4(v[0]);
        // which sum this lane holds: one bit a split, from the first split (xor 32) down
        constexpr uint32_t kSplits = kSums == 8u ? 3u : 2u;
        const uint32_t mine = lane >> (6u - kSplits);
        if ((lane & ((64u >> kSplits) - 1u)) == 0u) {
            const uint32_t u = mine / uint32_t(ROWS), r = mine % uint32_t(ROWS);
            if (t + u < t1 && e0 + r < num_experts) logits[size_t(t + u) * num_experts + e0 + r] = v[0];
        }
    };
    uint4 staged[TPS][kStage][Q];  // live across a step's arithmetic; handed to the lambdas as a parameter so it stays in registers
    stage_load(staged, t0);
    stage_store(staged, 0);
    __syncthreads();
    uint32_t buf = 0;
    for (uint32_t t = t0; t < t1; t += TPS, buf ^= 1u) {
        const bool more = t + TPS < t1;
        if (more) stage_load(staged, t + TPS);
        step(buf, t);
        if (more) stage_store(staged, buf ^ 1u);
        __syncthreads();
    }
}

// ---- the same logits on the matrix cores, for many tokens
//
// v_mfma_f32_16x16x1_4b_f32 is, in each of its four blocks, one IEEE multiply-add an output (checked against fmaf over
// subnormal products, cancellations and all exponents: the same bits), so a chain of them adds what a lane of router_row adds,
// in its order. A block's chain is one of router_row's 64 lanes: an output's lane sums l = p + 16 b, b = 0 .. 3, are the four
// blocks of one accumulator over chunks l, l + 64, ...; the first two stages of the butterfly (xor 32, 16) add the blocks, the
// next two (8, 4) the accumulators of p = 4 j + w, j = 0 .. 3, that wave w goes through, and the last two (2, 1) meet the four
// waves in LDS. An affine row's chunk sums its codes' products from zero, in 8 or 16 chains of their own, and takes scale
// (a multiply-add an output) and bias (one more MFMA) as router_row does.
//
// A workgroup takes 16 tokens and 16 experts, up to four workgroups a compute unit (three of 8-bit rows past 3,264 and of 4-bit ones
// past 1,536, two of 4-bit ones past 2,688: LogitsLds). Both sides' chunks come through a ring in LDS, a walk
// (four chunks of each wave's) a unit, asked for one or two units ahead. The effective scales come that way too and are widened
// in LDS once. What bounds it: a SIMD does not run a fp32 matrix instruction beside a vector one (a chain of them fed by two
// vector instructions each, two waves a SIMD: 44 cycles a step, 32 without), so 4,096 tokens of 2,048 against 256 rows, 28 us
// of matrix instructions alone, take 45 with the two conversions a product that nothing shares, and more with the loads' addresses.
// A step's chunks all asked for, waited for and multiplied by turns -> the ring, us: fp16 rows, 256 of 2,048: 512 tokens 13.2 ->
// 12.4, 1,000 21.0 -> 19.7, 4,096 69.5 -> 67.0, 128 of 3,072, 2,048 tokens 33.8 -> 26.9; 8-bit rows, 256 of 2,304: 300 tokens 18.4 ->
// 17.8, 1,000 34.1 -> 30.7, 2,000 60.0 -> 55.9; 4-bit rows, 1,000 tokens: 256 of 1,024 21.9 -> 20.7, of 1,600 22.2 -> 22.6, of 2,048 22.4 -> 21.7,
// 128 of 4,096, 2,000 tokens 47.1 -> 43.5. A place more each: 3 to 8 % slower past 1,000 tokens (a workgroup
// fewer a compute unit). Two tiles of tokens, or of experts, a workgroup: 512 tokens 13.5, 4,096 71 (half the workgroups); two of both spill.
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// PIECES: the effective scales start at a whole piece of 16 bytes; else they are loaded one by one (an instance of its own: the
// question alone cost the fp16 kernel 1 to 3 %).
template <int RK, bool PIECES>
__global__ __launch_bounds__(256, 4) void k_prefill_logits_mfma(RouterArgs a, uint32_t query_count, uint32_t stride, float *logits) {
    warm_kernel_arguments(a);
    typedef LogitsLds<RK> L;
    constexpr uint32_t E = kRouterChunk<RK>, Q = L::kPieces;  // a chunk's elements, 16-byte pieces of x
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t lane = threadIdx.x & 63u, wave = wave_index();
    const uint32_t num_experts = a.sel.num_experts, d = a.d, chunks = d / E, walks = (chunks + 63u) / 64u, groups = d / kGroup;
    // an XCD takes token tiles with all their expert tiles: the rows of `hidden` come to one L2, the experts' to every one
    const uint32_t expert_tiles = (num_experts + 15u) / 16u;
    const uint32_t t0 = ((blockIdx.x >> 3) / expert_tiles * 8u + (blockIdx.x & 7u)) * 16u, e0 = (blockIdx.x >> 3) % expert_tiles * 16u;
    if (t0 >= query_count) return;
    const uint32_t blocks = L::blocks(d), unit_bytes = L::unit(d);
    float *l_eff = reinterpret_cast<float *>(lds + L::eff(d));
    uint16_t *l_scale = reinterpret_cast<uint16_t *>(l_eff + d), *l_bias = l_scale + 16u * groups;
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)lds));
    // the effective scales as they are, into the last place, for now
    const uint32_t eff_at = (L::kPlaces - 1u) * unit_bytes;  // (2 d bytes: at most what the chunks of x take there)
    for (uint32_t i = wave * 1024u; PIECES && i < 2u * d; i += 4096u)
        lds_load16(lds0 + eff_at + i, reinterpret_cast<const uint8_t *>(a.effective_scale) + min(i + lane * 16u, 2u * d - 16u));
    // A load brings a 16-byte piece of four chunks of sixteen rows, the chunks xor-ed with the row so that sixteen rows read
    // at one chunk touch every bank once. Wave w brings block w's.
    const uint32_t l_row = lane >> 2, l_chunk = ((lane & 3u) ^ ((l_row >> 2) & 3u)) + 16u * wave;
    const uint8_t *w_row = static_cast<const uint8_t *>(a.weights) + size_t(min(e0 + l_row, num_experts - 1u)) * chunks * 16u;
    const uint16_t *x_row = a.hidden + size_t(min(t0 + l_row, query_count - 1u)) * stride;
    auto order = [](uint32_t step) { return step == 1u ? 2u : step == 2u ? 1u : step; };  // of j: the butterfly's
    const uint32_t units = 4u * walks;
    uint32_t ask_j = 0, ask_i = 0, ask_place = 0;  // the unit to ask for next: its step, its walk, its place
    auto ask = [&]() {
        const uint32_t c = min(4u * order(ask_j) + l_chunk + 64u * ask_i, chunks - 1u), at = lds0 + ask_place * unit_bytes;  // past the row: a copy, taken as zero
        if (RK != 4 || wave < blocks) {  // (a wave of the others always has chunks, and the branch is not free: 4,096 fp16 tokens 67.5, 69.1 us)
#pragma unroll
            for (uint32_t q = 0; q < Q; ++q) lds_load16(at + (wave * Q + q) * 1024u, x_row + c * E + q * 8u);
            lds_load16(at + (blocks * Q + wave) * 1024u, w_row + c * 16u);
        }
        if (++ask_i == walks) {
            ask_i = 0;
            ++ask_j;
        }
        ask_place = ask_place + 1u == L::kPlaces ? 0u : ask_place + 1u;
    };
#pragma unroll
    for (uint32_t u = 0; u + 1u < L::kPlaces; ++u)
        if (u < units) ask();
    if (RK != 0) {
        for (uint32_t i = threadIdx.x; i < 16u * groups; i += 256u) {
            const uint32_t e = min(e0 + i / groups, num_experts - 1u);
            l_scale[i] = a.scales[size_t(e) * groups + i % groups];
            l_bias[i] = a.biases[size_t(e) * groups + i % groups];
        }
    }
    if (L::kPlaces - 2u < units) wait_loads_and_sync<int((L::kPlaces - 2u) * (Q + 1u))>();
    else wait_loads_and_sync<0>();
    for (uint32_t i = threadIdx.x; i < d / 8u; i += 256u) {
        alignas(16) uint16_t v[8];
        if (PIECES) {
            *reinterpret_cast<uint4 *>(v) = *reinterpret_cast<const uint4 *>(lds + eff_at + i * 16u);
        } else {
#pragma unroll
            for (uint32_t n = 0; n < 8u; ++n) v[n] = a.effective_scale[8u * i + n];
        }
        float4 *to = reinterpret_cast<float4 *>(l_eff + 8u * i);
        to[0] = make_float4(bf16_to_f32(v[0]), bf16_to_f32(v[1]), bf16_to_f32(v[2]), bf16_to_f32(v[3]));
        to[1] = make_float4(bf16_to_f32(v[4]), bf16_to_f32(v[5]), bf16_to_f32(v[6]), bf16_to_f32(v[7]));
    }
    const uint32_t m = lane & 15u, block = lane >> 4;
    const uint32_t read_at = m * 64u + ((wave ^ ((m >> 2) & 3u)) * 16u), held = min(block, blocks - 1u);  // (a block without chunks reads another's: zero)
    f32x16_t acc;
    // chunk 64 i + 4 j + wave of each block; CHECK: it may lie past the row
    auto chunk = [&](uint32_t place, uint32_t j, uint32_t i, auto check) {
        constexpr bool CHECK = decltype(check)::value;
        const uint32_t c0 = 4u * j + wave + 64u * i, c = c0 + 16u * block;
        const bool inside = !CHECK || c < chunks;
        const uint32_t cc = inside ? c : 0u;
        const uint8_t *unit = lds + place * unit_bytes + read_at;
        const uint4 wv = *reinterpret_cast<const uint4 *>(unit + (blocks * Q + held) * 1024u);
        uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
        if (CHECK) {
#pragma unroll
            for (int n = 0; n < 4; ++n) ww[n] = inside ? ww[n] : 0u;
        }
        f32x16_t part = {0};
        float sum = 0.0f;
#pragma unroll
        for (uint32_t q = 0; q < Q; ++q) {
            const uint4 xv = *reinterpret_cast<const uint4 *>(unit + (held * Q + q) * 1024u);
            const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w};
            const float4 e0v = *reinterpret_cast<const float4 *>(l_eff + cc * E + q * 8u), e1v = *reinterpret_cast<const float4 *>(l_eff + cc * E + q * 8u + 4u);
            const float ew[8] = {e0v.x, e0v.y, e0v.z, e0v.w, e1v.x, e1v.y, e1v.z, e1v.w};
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                // moe.metal:357-358 (the exact product; + 0 makes it one instruction, and a zero's sign is nothing to a sum
                // that starts at +0)
                // (past the row the product is the zero, not its factor: chunk 0's effective scale may be infinite)
                const float product = fmaf(f16_to_f32(uint16_t(xw[k / 2u] >> (16u * (k & 1u)))), ew[k], 0.0f), x = inside ? product : 0.0f;
                if (RK == 0) {
                    acc = __builtin_amdgcn_mfma_f32_16x16x1f32(x, f16_to_f32(uint16_t(ww[k / 2u] >> (16u * (k & 1u)))), acc, 0, 0, 0);
                } else {
                    constexpr uint32_t kBits = RK == 0 ? 8u : uint32_t(RK), kPer = 32u / kBits;
                    const uint32_t n = q * 8u + k;
                    const float code = float((ww[n / kPer] >> (kBits * (n % kPer))) & ((1u << kBits) - 1u));
                    part = __builtin_amdgcn_mfma_f32_16x16x1f32(x, code, part, 0, 0, 0);
                    sum = __fadd_rn(sum, x);
                }
            }
        }
        if (RK != 0) {
#pragma unroll
            for (uint32_t b = 0; b < 4u; ++b) {
                const uint32_t cb = c0 + 16u * b;
                const float sc = !CHECK || cb < chunks ? meta_f32(l_scale[m * groups + cb * E / kGroup], a.meta) : 0.0f;
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r) acc[4u * b + r] = fmaf(sc, part[4u * b + r], acc[4u * b + r]);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(sum, inside ? meta_f32(l_bias[m * groups + cc * E / kGroup], a.meta) : 0.0f, acc, 0, 0, 0);
        }
    };
    float even[4], odd[4];
    uint32_t unit = 0, place = L::kPlaces - 1u;
    // The place of the next unit: it has landed for every wave, and every wave is done with the one before it, whose place is asked
    // for again.
    auto take = [&]() {
        if (unit + L::kPlaces - 2u < units) wait_loads_and_sync<int((L::kPlaces - 2u) * (Q + 1u))>();
        else wait_loads_and_sync<0>();
        if (unit + L::kPlaces - 1u < units) ask();
        ++unit;
        place = place + 1u == L::kPlaces ? 0u : place + 1u;
        return place;
    };
#pragma unroll
    for (uint32_t step = 0; step < 4u; ++step) {
        acc = f32x16_t{0};
        // (the walk that may end past the row is on its own: in one loop with the others the sums went from register to register)
        for (uint32_t i = 0; i + 1u < walks; ++i) chunk(take(), order(step), i, std::false_type{});
        const uint32_t last = take();
        if (64u * walks == chunks) chunk(last, order(step), walks - 1u, std::false_type{});
        else chunk(last, order(step), walks - 1u, std::true_type{});
#pragma unroll
        for (uint32_t r = 0; r < 4u; ++r) {
            const float v = __fadd_rn(__fadd_rn(acc[r], acc[8u + r]), __fadd_rn(acc[4u + r], acc[12u + r]));
            if (step == 0u) even[r] = v;
            else if (step == 1u) even[r] = __fadd_rn(even[r], v);
            else if (step == 2u) odd[r] = v;
            else even[r] = __fadd_rn(even[r], __fadd_rn(odd[r], v));
        }
    }
    __syncthreads();  // (nobody reads the operands any more)
    float (*meet)[16][17] = reinterpret_cast<float (*)[16][17]>(lds);
    static_assert(sizeof(float[4][16][17]) <= L::kPlaces * L::kBlock, "the waves' sums fit where the smallest units were");
#pragma unroll
    for (uint32_t r = 0; r < 4u; ++r) meet[wave][4u * block + r][m] = even[r];
    __syncthreads();
    const uint32_t row = threadIdx.x >> 4, col = threadIdx.x & 15u;
    const float v = __fadd_rn(__fadd_rn(meet[0][row][col], meet[2][row][col]), __fadd_rn(meet[1][row][col], meet[3][row][col]));
    if (t0 + row < query_count && e0 + col < num_experts) logits[size_t(t0 + row) * num_experts + e0 + col] = v;
}

// True if it launched: where 16 tokens by 16 experts make more than one workgroup for most compute units. With fewer a workgroup's
// chain of units is what it takes, some 8 us, and the vector kernel's many small workgroups are done before (fp16 rows,
// 256 of 2,048: 300 tokens 16.3 against 15.4 us with the selection, 512 17.3 against 20.2; 8-bit, 2,304: 100 tokens 17.1
// against 16.2, 300 22.3 against 24.2).
template <int RK>
static bool launch_prefill_logits_mfma(const RouterArgs &a, uint32_t query_count, uint32_t stride, float *logits, hipStream_t s) {
    const uint32_t expert_tiles = (a.sel.num_experts + 15u) / 16u, token_tiles = (query_count + 15u) / 16u;
    if (uint64_t(expert_tiles) * token_tiles <= (RK == 0 ? 384u : 256u)) return false;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(((token_tiles + 7u) & ~7u) * expert_tiles), dim3(256), LogitsLds<RK>::bytes(a.d), s, a, query_count, stride, logits);
    };
    // (scales at an odd element, us with the selection, on the vector kernel and here: 4,096 tokens of 2,048 against 256 rows 85, 65;
    // 8-bit rows, 1,000 of 2,304, 48, 32)
    if (reinterpret_cast<uintptr_t>(a.effective_scale) % 16u == 0) launch(k_prefill_logits_mfma<RK, true>);
    else launch(k_prefill_logits_mfma<RK, false>);
    return true;
}

template <int RK, int MAXC, int ROWS>
static void launch_prefill_logits(const RouterArgs &a, uint32_t query_count, uint32_t stride, float *logits, hipStream_t s) {
    constexpr uint32_t kStepTokens = 2;
    const uint32_t blocks = (a.sel.num_experts + 4u * ROWS - 1u) / (4u * ROWS);
    // Tokens a workgroup walks with its rows: as few as a step takes while that still leaves the chip short of workgroups
    // (37 tokens, 256 rows: 9.1 us with 2, 11.7 with 8), more where there are plenty, since a workgroup first fetches its
    // rows (4,096 tokens: 114 us with 2, 94 with 4, 87 with 8 and 16; past 16 the last wave of workgroups costs more).
    uint32_t tokens = kStepTokens;
    while (tokens < 16u && blocks * ((query_count + tokens - 1u) / tokens) > 1280u) tokens *= 2u;
    hipLaunchKernelGGL((k_prefill_logits<RK, MAXC, ROWS, kStepTokens>), dim3(blocks, (query_count + tokens - 1u) / tokens), dim3(256),
                       0, s, a, query_count, stride, logits, tokens);
}

// prefill.metal:441-563: one wave selects for one token.
// group_sums (may be null): the wave also leaves, for its token's row of `hidden`, the sum of every group of 64 of its fp16
// elements, exactly as k_row_group_sums forms it (a lane takes an 8-element chunk: its eight values in order, then eight
// neighbouring lanes fold pairwise), as (hi, lo) halves at [token][group]. The launch is a chain of dependent steps on half the
// chip's compute units: the row's loads go out ahead of the selection and are summed behind it.
template <bool SUMS>
__global__ __launch_bounds__(256) void k_prefill_select(SelectArgs sel, const float *ws, uint32_t *out_indices,
                                                        uint16_t *out_weights, uint32_t query_count, const uint16_t *hidden,
                                                        uint32_t stride, uint32_t d, uint32_t *group_sums) {
    warm_kernel_arguments(sel);
    __shared__ RouteScratch s_route[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t t = blockIdx.x * 4u + wave;
    if (t >= query_count) return;
    constexpr uint32_t kAhead = SHRIKE_MAX_HIDDEN / 8u / 64u;  // chunks a lane can own
    uint4 mine[SUMS ? kAhead : 1u];
    const uint32_t chunks = d / 8u;
    if (SUMS) {
        const uint4 *row = reinterpret_cast<const uint4 *>(hidden + size_t(t) * stride);
#pragma unroll
        for (uint32_t i = 0; i < kAhead; ++i)
            if (64u * i < chunks) mine[i] = row[min(lane + 64u * i, chunks - 1u)];  // past the row: a copy, never stored
    }
    sel.logits = ws + size_t(t) * sel.num_experts;
    RouteLists lists = {};
    lists.out_indices = out_indices + size_t(t) * sel.top_k;
    lists.out_weights = out_weights + size_t(t) * sel.top_k;
    uint32_t cell;
    route_wave<false>(sel, lists, lane, true, cell, s_route[wave]);
    if (SUMS) {
#pragma unroll
        for (uint32_t i = 0; i < kAhead; ++i) {
            if (64u * i >= chunks) break;
            const uint32_t c = lane + 64u * i;
            const uint32_t xw[4] = {mine[i].x, mine[i].y, mine[i].z, mine[i].w};
            float sum = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                sum = __fadd_rn(sum, f16_to_f32(uint16_t(xw[q])));
                sum = __fadd_rn(sum, f16_to_f32(uint16_t(xw[q] >> 16)));
            }
            sum = butterfly_of_8(sum);
            if (c < chunks && (c & 7u) == 0u) group_sums[size_t(t) * (d / 64u) + (c >> 3)] = split_hi_lo(sum);  // d % 64 == 0: whole groups
        }
    }
}

// ---- grouping ---------------------------------------------------------------------------

struct GroupArgs {
    const uint32_t *indices;
    const uint16_t *weights;
    uint32_t pairs, top_k, num_experts;
    const uint64_t *sort_keys, *residency;
    shrike_token_expert_pair *sorted;
    uint32_t *offsets, *counts;
    shrike_row_tile *tiles;
    uint32_t *tile_count;
};

constexpr uint32_t kGroupLdsPairs = 131072;   // pairs whose expert ids (one byte each) fit the LDS copy
constexpr uint32_t kGroupLdsWeights = 49152;  // pairs whose fp16 weights are staged beside them

// One launch, four experts a workgroup (one a wave). Every workgroup builds the whole
// histogram for itself in LDS (the pairs are a few KB and sit in L2), so no count has to
// cross workgroups. A wave then knows its expert's first position (the pairs of every
// expert ordered before it), writes its row tiles, and writes its pairs in index order.
// The pairs arrive token-major, so index order is (token, rank) order: the permutation
// equals the reference's sort by (sort key, expert, token, rank)
// (PrefillMoEGrouping.swift:323-332).
//
// PARTS: the pairs are cut into as many runs, each with 256 threads and a histogram of its own, and an expert's pairs of a run
// are placed by a wave of its own, behind those of the runs before. All of it is latency, of the pairs' loads and of the
// placement's steps: with four runs instead of one, and every pair's weight in LDS beside its id, 32,768 pairs over 256
// experts take 15 us where they took 35, 8,000 take 8 where they took 11.
template <uint32_t PARTS>
__global__ __launch_bounds__(256 * PARTS) void k_group(GroupArgs a) {
    warm_kernel_arguments(a);
    extern __shared__ __align__(16) uint8_t s_group[];
    uint32_t (*s_hist)[SHRIKE_MAX_ROUTER_EXPERTS] = reinterpret_cast<uint32_t (*)[SHRIKE_MAX_ROUTER_EXPERTS]>(s_group);
    uint8_t *s_ids = s_group + PARTS * SHRIKE_MAX_ROUTER_EXPERTS * 4u;
    uint16_t *s_weights = reinterpret_cast<uint16_t *>(s_ids + ((a.pairs + 15u) & ~15u));
    const uint32_t part = threadIdx.x >> 8, in_part = threadIdx.x & 255u;
    const uint32_t part_pairs = ((a.pairs + PARTS - 1u) / PARTS + 15u) & ~15u;  // (whole 16-byte reads of ids)
    const uint32_t lo = min(part * part_pairs, a.pairs), hi = min(lo + part_pairs, a.pairs);
    const bool in_lds = a.pairs <= kGroupLdsPairs;
    // the placement loop below is one dependent step a 64 pairs: a global load inside it would
    // cost its full latency every step
    const bool weights_in_lds = a.pairs <= kGroupLdsWeights;
    s_hist[part][in_part] = 0u;
    __syncthreads();
    // sixteen pairs a thread at a time: all their loads go out before the first is used (with the uses
    // inside the loading loop every load was waited for on the spot, thirty-two round trips to L2 on end)
    constexpr uint32_t kPairsAThread = 16;
    for (uint32_t base = lo; base < hi; base += 256u * kPairsAThread) {
        uint32_t v[kPairsAThread];
        uint16_t wv[kPairsAThread];
#pragma unroll
        for (uint32_t j = 0; j < kPairsAThread; ++j) {
            const uint32_t i = min(base + j * 256u + in_part, a.pairs - 1u);
            v[j] = a.indices[i];
            wv[j] = a.weights[i];
        }
#pragma unroll
        for (uint32_t j = 0; j < kPairsAThread; ++j) {
            const uint32_t i = base + j * 256u + in_part;
            if (i >= hi) continue;
            if (v[j] < a.num_experts) atomicAdd(&s_hist[part][v[j]], 1u);
            if (in_lds) s_ids[i] = uint8_t(min(v[j], 255u));
            if (weights_in_lds) s_weights[i] = wv[j];
        }
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, e = blockIdx.x * 4u + (in_part >> 6);
    if (e >= a.num_experts) return;
    // the keys and the residency word are fetched together, ahead of their use
    const uint64_t key = a.sort_keys ? a.sort_keys[e] : 0u;
    const uint64_t word = a.residency ? a.residency[e] : 0u;
    uint64_t other_key[SHRIKE_MAX_ROUTER_EXPERTS / 64u];
#pragma unroll
    for (uint32_t j = 0; j < SHRIKE_MAX_ROUTER_EXPERTS / 64u; ++j)
        other_key[j] = a.sort_keys ? a.sort_keys[min(lane + 64u * j, a.num_experts - 1u)] : 0u;
    uint32_t offset = 0, tiles_before = 0, tiles_total = 0;
#pragma unroll
    for (uint32_t j = 0; j < SHRIKE_MAX_ROUTER_EXPERTS / 64u; ++j) {
        const uint32_t other = lane + 64u * j;
        if (other >= a.num_experts) continue;
        uint32_t c = s_hist[0][other];
#pragma unroll
        for (uint32_t q = 1; q < PARTS; ++q) c += s_hist[q][other];
        const uint64_t k2 = other_key[j];
        const bool before = k2 < key || (k2 == key && other < e);
        const uint32_t t = (c + kRowTile - 1u) / kRowTile;
        offset += before ? c : 0u;
        tiles_before += before ? t : 0u;
        tiles_total += t;
    }
    offset = wave_sum_u32(offset);
    tiles_before = wave_sum_u32(tiles_before);
    tiles_total = wave_sum_u32(tiles_total);
    uint32_t count = 0, ahead = 0;  // of the expert's pairs, and those in the runs before this one
#pragma unroll
    for (uint32_t q = 0; q < PARTS; ++q) {
        ahead += q < part ? s_hist[q][e] : 0u;
        count += s_hist[q][e];
    }
    if (lane == 0 && part == 0u) {
        a.counts[e] = count;
        a.offsets[e] = count ? offset : 0xffffffffu;
        if (e == 0) *a.tile_count = tiles_total;
    }
    uint32_t cell = e;
    if (a.residency)  // moe.metal:136-146
        cell = uint32_t(word >> 32) == SHRIKE_RESIDENCY_RESIDENT ? uint32_t(word) : kSentinel;
    const uint32_t my_tiles = (count + kRowTile - 1u) / kRowTile;
    for (uint32_t j = part * 64u + lane; j < my_tiles; j += PARTS * 64u) {
        shrike_row_tile t;
        t.cell = cell;
        t.pair_start = offset + j * kRowTile;
        t.rows = min(kRowTile, count - j * kRowTile);
        t.expert = e;
        a.tiles[tiles_before + j] = t;
    }
    const uint32_t here = s_hist[part][e];
    if (here == 0) return;
    offset += ahead;
    // i / top_k == umulhi(i, magic) for i * top_k < 2^32; top_k == 1 would need magic 2^32, so it divides plainly below
    const uint32_t token_magic = 0xffffffffu / a.top_k + 1u;
    uint32_t running = 0;
    if (in_lds) {
        // 1,024 pairs a step: a lane takes 16 neighbouring ids with one LDS read, flags the bytes equal
        // to e, and a prefix sum over the lanes turns the per-lane counts into positions in index order
        const uint32_t pattern = e * 0x01010101u;
        for (uint32_t base = lo; base < hi && running < here; base += 1024u) {
            const uint32_t i0 = base + lane * 16u;
            uint32_t match = 0;
            if (i0 < hi) {
                const uint4 v = *reinterpret_cast<const uint4 *>(s_ids + i0);
                const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t x = words[w] ^ pattern;  // a zero byte where the id is e
                    const uint32_t t = ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu);  // 0x80 in exactly those bytes
                    match |= ((((t >> 7) * 0x01020408u) >> 24) & 0xfu) << (4 * w);
                }
                const uint32_t valid = hi - i0;  // ids past the last pair are whatever the LDS held
                if (valid < 16u) match &= (1u << valid) - 1u;
            }
            const uint32_t mine = __popc(match);
            const uint32_t upto = wave_inclusive_scan_u32(mine);
            uint32_t at = offset + running + upto - mine;
            while (match) {
                const uint32_t i = i0 + uint32_t(__ffs(int(match)) - 1);
                match &= match - 1u;
                shrike_token_expert_pair p;
                p.token = a.top_k == 1u ? i : __umulhi(i, token_magic);
                p.expert = e;
                p.rank = i - p.token * a.top_k;
                p.weight_bits_and_reserved = weights_in_lds ? s_weights[i] : a.weights[i];
                if (at < offset + here) a.sorted[at] = p;  // ids the histogram did not count (out of range) never land
                ++at;
            }
            running += uint32_t(__builtin_amdgcn_readlane(int(upto), 63));
        }
        return;
    }
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    for (uint32_t base = lo; base < hi && running < here; base += 64u) {
        const uint32_t i = base + lane;
        const bool mine = i < hi && a.indices[i] == e;
        const uint64_t mask = __ballot(mine);
        if (mine) {
            shrike_token_expert_pair p;
            p.token = a.top_k == 1u ? i : __umulhi(i, token_magic);
            p.expert = e;
            p.rank = i - p.token * a.top_k;
            p.weight_bits_and_reserved = a.weights[i];
            a.sorted[offset + running + __popcll(mask & below)] = p;
        }
        running += __popcll(mask);
    }
}

// ---- group sums -------------------------------------------------------------------------

// For every row of an fp16 matrix [rows, n] (row r at r * stride), the sum of each group of
// 64 elements, accumulated in fp32 in a fixed order and stored as two fp16 halves (hi, lo):
// the operand that turns the affine bias term sum_g bias[g] * (sum of x over g) into one
// more matrix product. Eight lanes share a group; a lane sums its eight elements in order,
// then the eight partials fold pairwise.
__global__ __launch_bounds__(256) void k_row_group_sums(const uint16_t *src, size_t stride, uint32_t rows, uint32_t n,
                                                        uint32_t *out, const uint32_t *row_limit_tiles) {
    const uint32_t groups = n / kGroup;
    const size_t slot = size_t(blockIdx.x) * 256u + threadIdx.x;  // (row, group, eighth)
    const size_t per_row = size_t(groups) * 8u;
    const uint32_t row = uint32_t(slot / per_row);
    uint32_t live_rows = rows;
    if (row_limit_tiles) live_rows = min(rows, *row_limit_tiles * kRowTile);
    const bool on = row < live_rows;
    const uint32_t rest = uint32_t(slot - size_t(row) * per_row);
    float s = 0.0f;
    if (on) {
        const uint4 v = *reinterpret_cast<const uint4 *>(src + size_t(row) * stride + size_t(rest) * 8u);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            s = __fadd_rn(s, f16_to_f32(uint16_t(w[t])));
            s = __fadd_rn(s, f16_to_f32(uint16_t(w[t] >> 16)));
        }
    }
    s = butterfly_of_8(s);
    if (on && (rest & 7u) == 0u) out[size_t(row) * groups + rest / 8u] = split_hi_lo(s);
}

// ---- reduce and residual ----------------------------------------------------------------

// prefill.metal:624-645: a thread owns eight neighbouring d of one token; fp32 fma in rank order
__global__ __launch_bounds__(256) void k_prefill_reduce(const uint16_t *partials, const uint16_t *weights, uint16_t *h2,
                                                        uint32_t query_count, uint32_t top_k, uint32_t d) {
    const uint32_t per_row = d / 8u;
    const size_t slot = size_t(blockIdx.x) * 256u + threadIdx.x;
    const uint32_t t = uint32_t(slot / per_row);
    if (t >= query_count) return;
    const uint32_t c = uint32_t(slot - size_t(t) * per_row);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (uint32_t r = 0; r < top_k; ++r) {
        const float w = f16_to_f32(weights[size_t(t) * top_k + r]);
        const uint4 v = *reinterpret_cast<const uint4 *>(partials + (size_t(t) * top_k + r) * d + size_t(c) * 8u);
        const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[2 * j] = fmaf(w, f16_to_f32(uint16_t(p[j])), acc[2 * j]);
            acc[2 * j + 1] = fmaf(w, f16_to_f32(uint16_t(p[j] >> 16)), acc[2 * j + 1]);
        }
    }
    uint4 o;
    o.x = uint32_t(f32_to_f16(acc[0])) | uint32_t(f32_to_f16(acc[1])) << 16;
    o.y = uint32_t(f32_to_f16(acc[2])) | uint32_t(f32_to_f16(acc[3])) << 16;
    o.z = uint32_t(f32_to_f16(acc[4])) | uint32_t(f32_to_f16(acc[5])) << 16;
    o.w = uint32_t(f32_to_f16(acc[6])) | uint32_t(f32_to_f16(acc[7])) << 16;
    *reinterpret_cast<uint4 *>(h2 + size_t(t) * d + size_t(c) * 8u) = o;
}

__global__ __launch_bounds__(256) void k_residual_add(uint16_t *hidden, const uint16_t *delta, uint64_t count) {
    const uint64_t i = (uint64_t(blockIdx.x) * 256u + threadIdx.x) * 8u;
    if (i >= count) return;
    if (i + 8u <= count) {
        uint4 h = *reinterpret_cast<const uint4 *>(hidden + i);
        const uint4 dl = *reinterpret_cast<const uint4 *>(delta + i);
        uint32_t hw[4] = {h.x, h.y, h.z, h.w};
        const uint32_t dw[4] = {dl.x, dl.y, dl.z, dl.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint16_t lo = f32_to_f16(__fadd_rn(f16_to_f32(uint16_t(hw[j])), f16_to_f32(uint16_t(dw[j]))));
            const uint16_t hi = f32_to_f16(__fadd_rn(f16_to_f32(uint16_t(hw[j] >> 16)), f16_to_f32(uint16_t(dw[j] >> 16))));
            hw[j] = uint32_t(lo) | uint32_t(hi) << 16;
        }
        h.x = hw[0]; h.y = hw[1]; h.z = hw[2]; h.w = hw[3];
        *reinterpret_cast<uint4 *>(hidden + i) = h;
    } else {
        for (uint64_t j = i; j < count; ++j) hidden[j] = f32_to_f16(__fadd_rn(f16_to_f32(hidden[j]), f16_to_f32(delta[j])));
    }
}

// shared_scalar_gate_rows, moe.metal:1154-1193: one 8-bit group-affine weight row against a block of token rows,
// a workgroup a row or ROWS of them. Eight partial sums as in the reference (its eight simdgroups of 32 lanes are the half-waves
// here): partial p takes the groups p, p + 8, ..., lane l of its 32 the elements 2l and 2l + 1 of a group; the 32
// lane sums fold by the butterfly 1, 2, 4, 8, 16 and the eight partials are added in index order.
// Bound by a workgroup's chain (loads, sums, barrier) and how many fit the chip: with many rows a workgroup takes several side by
// side, the weights' codes and scales read once for them (4,096 rows of 2,048 in a chunk's pass: 8.3 us with a row a workgroup, 6.0
// with four).
template <uint32_t ROWS>
__global__ __launch_bounds__(256) void k_scalar_gate_rows(const uint8_t *w, const uint16_t *scales, const uint16_t *biases,
                                                          uint32_t meta, const uint16_t *x, uint32_t x_stride, uint16_t *gate,
                                                          uint32_t d, uint32_t rows) {
    __shared__ float s_partial[ROWS][8];
    const uint32_t p = threadIdx.x >> 5, l = threadIdx.x & 31u;
    const uint16_t *row[ROWS];
    float acc[ROWS];
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
        row[r] = x + size_t(min(blockIdx.x * ROWS + r, rows - 1u)) * x_stride;  // (past the last row: a copy, not stored)
        acc[r] = 0.0f;
    }
    for (uint32_t g = p; g < d / kGroup; g += 8u) {
        const uint32_t i0 = g * kGroup + 2u * l;
        uint32_t xw[ROWS];
#pragma unroll
        for (uint32_t r = 0; r < ROWS; ++r) xw[r] = *reinterpret_cast<const uint32_t *>(row[r] + i0);
        const uint16_t qw = *reinterpret_cast<const uint16_t *>(w + i0);
        const float scale = meta_f32(scales[g], meta), bias = meta_f32(biases[g], meta);
#pragma unroll
        for (uint32_t r = 0; r < ROWS; ++r) {
            const float x0 = f16_to_f32(uint16_t(xw[r])), x1 = f16_to_f32(uint16_t(xw[r] >> 16));
            const float dot = __fadd_rn(__fmul_rn(float(qw & 0xffu), x0), __fmul_rn(float(qw >> 8), x1));
            acc[r] = fmaf(scale, dot, acc[r]);
            acc[r] = fmaf(bias, __fadd_rn(x0, x1), acc[r]);
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
        acc[r] = butterfly_of_32(acc[r]);
        if (l == 0) s_partial[r][p] = acc[r];
    }
    __syncthreads();
    const uint32_t mine = blockIdx.x * ROWS + threadIdx.x;
    if (threadIdx.x < ROWS && mine < rows) {
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) total = __fadd_rn(total, s_partial[threadIdx.x][i]);
        gate[mine] = f32_to_f16(total);
    }
}

// sigmoid_scalar_mul_rows_fp16, moe.metal:1195-1207: y[row, i] = half(y[row, i] / (1 + exp(-gate[row]))), eight
// elements a thread.
__global__ __launch_bounds__(256) void k_sigmoid_scalar_mul_rows(uint16_t *y, const uint16_t *gate, uint32_t d, uint32_t rows) {
    const uint32_t per_row = d / 8u;
    const uint64_t slot = uint64_t(blockIdx.x) * 256u + threadIdx.x;
    if (slot >= uint64_t(rows) * per_row) return;
    const uint32_t r = uint32_t(slot / per_row);
    const float div = 1.0f + expf(-f16_to_f32(gate[r]));
    uint4 v = *reinterpret_cast<const uint4 *>(y + slot * 8u);
    uint32_t vw[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint16_t lo = f32_to_f16(f16_to_f32(uint16_t(vw[j])) / div);
        const uint16_t hi = f32_to_f16(f16_to_f32(uint16_t(vw[j] >> 16)) / div);
        vw[j] = uint32_t(lo) | uint32_t(hi) << 16;
    }
    v.x = vw[0]; v.y = vw[1]; v.z = vw[2]; v.w = vw[3];
    *reinterpret_cast<uint4 *>(y + slot * 8u) = v;
}

int launch_row_group_sums(const uint16_t *src, size_t stride, uint32_t rows, uint32_t n, uint32_t *out,
                          const uint32_t *row_limit_tiles, hipStream_t s) {
    const size_t slots = size_t(rows) * (n / kGroup) * 8u;
    if (slots == 0) return 0;
    hipLaunchKernelGGL(k_row_group_sums, dim3(uint32_t((slots + 255u) / 256u)), dim3(256), 0, s, src, stride, rows, n, out,
                       row_limit_tiles);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

}  // namespace shrike

using namespace shrike;

// d_group_sums (may be null): where the group sums of hidden's rows go as well, for the grouped FFN's bias term
static int prefill_router(shrike_hip_moe *moe, void *stream, const void *d_weights, const void *d_scales, const void *d_biases,
                          const void *d_hidden, const void *d_effective_scale, const void *d_per_expert_scale,
                          const void *d_logit_bias, uint32_t *d_out_indices, void *d_out_weights, float *d_logits_workspace,
                          uint32_t query_count, uint32_t num_experts, uint32_t d, uint32_t top_k, uint32_t hidden_stride_elements,
                          uint32_t *d_group_sums) {
    SHRIKE_REQUIRE(moe != nullptr, "moe handle is NULL");
    SHRIKE_REQUIRE(query_count > 0, "queryCount must be positive");  // PrefillRouter.swift:99
    if (int rc = check_router(moe, num_experts, d, top_k)) return rc;
    SHRIKE_REQUIRE(hidden_stride_elements >= d, "hidden stride is too small");  // PrefillRouter.swift:104
    SHRIKE_REQUIRE(hidden_stride_elements % 8u == 0, "hidden stride must keep rows 16-byte aligned");
    SHRIKE_REQUIRE(d_weights && d_hidden && d_effective_scale && d_per_expert_scale && d_logit_bias,
                   "prefill router: weights, hidden, effectiveScale, perExpertScale and logitBias must all be bound");
    SHRIKE_REQUIRE(moe->desc.router_weight_bits == 0 || (d_scales && d_biases), "prefill router: affine router needs scales and biases");
    SHRIKE_REQUIRE(d_out_indices && d_out_weights && d_logits_workspace, "prefill router: outputs and the workspace must be bound");
    SHRIKE_REQUIRE(reinterpret_cast<uintptr_t>(d_logits_workspace) % 16u == 0, "prefill router: workspace must be 16-byte aligned");
    RouterArgs a = {};
    a.weights = d_weights;
    a.scales = static_cast<const uint16_t *>(d_scales);
    a.biases = static_cast<const uint16_t *>(d_biases);
    a.hidden = static_cast<const uint16_t *>(d_hidden);
    a.effective_scale = static_cast<const uint16_t *>(d_effective_scale);
    a.d = d;
    a.meta = moe->desc.meta_dtype;
    a.sel.per_expert_scale = static_cast<const uint16_t *>(d_per_expert_scale);
    a.sel.logit_bias = static_cast<const uint16_t *>(d_logit_bias);
    a.sel.num_experts = num_experts;
    a.sel.top_k = top_k;
    a.sel.sigmoid = moe->desc.sigmoid_router_scores;
    a.sel.scaling = moe->desc.routed_scaling_factor;
    hipStream_t s = as_stream(stream);
    // A few tokens over a few experts: the decode router's kernel with the tokens on the grid, one launch for logits and
    // selection. Past about 512 rows in all its workgroups (a row a wave, the rows fetched again for every token) cost more
    // than a second launch (256 rows: 2 tokens 7.3 against 6.9 us, 8 tokens 11.4 against 7.2), and where the group sums are
    // wanted too it would need a second launch anyway; of affine rows the two launches widen every code first, which one or
    // two tokens do not pay back (8.8 against 9.7 us).
    const bool few_rows = uint64_t(query_count) * num_experts <= 512u && query_count <= kRouterLaunchTokens;
    if (few_rows && (d_group_sums == nullptr || (moe->desc.router_weight_bits != 0 && query_count <= 2u))) {
        a.logits_out = d_logits_workspace;
        a.sel.logits = d_logits_workspace;
        a.lists.out_indices = d_out_indices;
        a.lists.out_weights = static_cast<uint16_t *>(d_out_weights);
        a.counter = moe->d_counter + kRouterTokenCounters;
        a.token_stride = hidden_stride_elements;
        if (int rc = launch_router_tokens(a, moe->desc.router_weight_bits, query_count, s)) return rc;
        return d_group_sums ? launch_row_group_sums(a.hidden, hidden_stride_elements, query_count, d, d_group_sums, nullptr, s) : 0;
    }
    // the vector kernel with as many rows a wave as their registers allow: four where a lane's share of a row is up to 48
    // elements, else two
    switch (moe->desc.router_weight_bits) {
        case 0:
            if (launch_prefill_logits_mfma<0>(a, query_count, hidden_stride_elements, d_logits_workspace, s)) break;
            if (d <= 2048u) launch_prefill_logits<0, 4, 4>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            else if (d <= 3072u) launch_prefill_logits<0, 6, 4>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            else launch_prefill_logits<0, 8, 2>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            break;
        case 8:
            if (launch_prefill_logits_mfma<8>(a, query_count, hidden_stride_elements, d_logits_workspace, s)) break;
            if (d <= 2048u) launch_prefill_logits<8, 2, 4>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            else if (d <= 3072u) launch_prefill_logits<8, 3, 4>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            else launch_prefill_logits<8, 4, 2>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            break;
        default:
            if (launch_prefill_logits_mfma<4>(a, query_count, hidden_stride_elements, d_logits_workspace, s)) break;
            if (d <= 2048u) launch_prefill_logits<4, 1, 4>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
            else launch_prefill_logits<4, 2, 2>(a, query_count, hidden_stride_elements, d_logits_workspace, s);
    }
    SHRIKE_HIP(hipGetLastError());
    if (d_group_sums)  // the selection's waves form them on the side
        hipLaunchKernelGGL(k_prefill_select<true>, dim3((query_count + 3u) / 4u), dim3(256), 0, s, a.sel, d_logits_workspace,
                           d_out_indices, static_cast<uint16_t *>(d_out_weights), query_count, a.hidden, hidden_stride_elements, d,
                           d_group_sums);
    else
        hipLaunchKernelGGL(k_prefill_select<false>, dim3((query_count + 3u) / 4u), dim3(256), 0, s, a.sel, d_logits_workspace,
                           d_out_indices, static_cast<uint16_t *>(d_out_weights), query_count, a.hidden, hidden_stride_elements, d,
                           nullptr);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

extern "C" {

int shrike_hip_prefill_router(shrike_hip_moe *moe, void *stream, const void *d_weights, const void *d_scales,
                              const void *d_biases, const void *d_hidden, const void *d_effective_scale,
                              const void *d_per_expert_scale, const void *d_logit_bias, uint32_t *d_out_indices,
                              void *d_out_weights, float *d_logits_workspace, uint32_t query_count, uint32_t num_experts,
                              uint32_t d, uint32_t top_k, uint32_t hidden_stride_elements) {
    return prefill_router(moe, stream, d_weights, d_scales, d_biases, d_hidden, d_effective_scale, d_per_expert_scale, d_logit_bias,
                          d_out_indices, d_out_weights, d_logits_workspace, query_count, num_experts, d, top_k,
                          hidden_stride_elements, nullptr);
}

int shrike_hip_prefill_router_with_group_sums(shrike_hip_moe *moe, void *stream, const void *d_weights, const void *d_scales,
                                              const void *d_biases, const void *d_hidden, const void *d_effective_scale,
                                              const void *d_per_expert_scale, const void *d_logit_bias,
                                              uint32_t *d_out_indices, void *d_out_weights, float *d_logits_workspace,
                                              uint32_t query_count, uint32_t num_experts, uint32_t d, uint32_t top_k,
                                              uint32_t hidden_stride_elements, void *d_ffn_workspace) {
    SHRIKE_REQUIRE(d_ffn_workspace != nullptr, "prefill router: the FFN workspace that takes the group sums is NULL");
    SHRIKE_REQUIRE(reinterpret_cast<uintptr_t>(d_ffn_workspace) % 256u == 0, "prefill router: the FFN workspace must be 256-byte aligned");
    SHRIKE_REQUIRE(d % kGroup == 0, "prefill router: group sums need d to be a multiple of 64, got %u", d);
    return prefill_router(moe, stream, d_weights, d_scales, d_biases, d_hidden, d_effective_scale, d_per_expert_scale, d_logit_bias,
                          d_out_indices, d_out_weights, d_logits_workspace, query_count, num_experts, d, top_k,
                          hidden_stride_elements, static_cast<uint32_t *>(d_ffn_workspace));
}

size_t shrike_hip_prefill_router_workspace_bytes(uint32_t query_count, uint32_t num_experts, uint32_t d) {
    (void)d;  // the fp32 logits alone: x times the effective scale is formed inside the logits kernel
    return ((size_t(query_count) * num_experts + 3u) & ~size_t(3)) * sizeof(float);
}

uint32_t shrike_hip_group_max_row_tiles(uint64_t pair_count, uint32_t num_experts) {
    return max_row_tiles(pair_count, num_experts);
}

int shrike_hip_group_pairs(void *stream, const uint32_t *d_indices, const void *d_weights, uint32_t query_count,
                           uint32_t top_k, uint32_t num_experts, const uint64_t *d_expert_sort_keys,
                           const uint64_t *d_residency, const shrike_hip_grouped_routes *out) {
    SHRIKE_REQUIRE(top_k > 0, "topK must be positive, got %u", top_k);                    // PrefillMoEGrouping.swift:280
    SHRIKE_REQUIRE(num_experts > 0, "numExperts must be positive, got %u", num_experts);  // :283
    SHRIKE_REQUIRE(num_experts <= SHRIKE_MAX_ROUTER_EXPERTS, "numExperts > 256 is not supported");
    SHRIKE_REQUIRE(uint64_t(query_count) * top_k <= 0x7fffffffull, "too many route pairs");
    SHRIKE_REQUIRE(out && out->sorted_pairs && out->per_expert_offsets && out->per_expert_counts && out->row_tiles && out->row_tile_count,
                   "group pairs: an output is NULL");
    SHRIKE_REQUIRE(query_count == 0 || (d_indices && d_weights), "group pairs: indices and weights must be bound");
    GroupArgs a = {};
    a.indices = d_indices;
    a.weights = static_cast<const uint16_t *>(d_weights);
    a.pairs = query_count * top_k;
    a.top_k = top_k;
    a.num_experts = num_experts;
    a.sort_keys = d_expert_sort_keys;
    a.residency = d_residency;
    a.sorted = static_cast<shrike_token_expert_pair *>(out->sorted_pairs);
    a.offsets = out->per_expert_offsets;
    a.counts = out->per_expert_counts;
    a.tiles = out->row_tiles;
    a.tile_count = out->row_tile_count;
    hipStream_t s = as_stream(stream);
    const dim3 grid((num_experts + 3u) / 4u);
    const uint32_t ids = (a.pairs + 15u) & ~15u;
    const uint32_t staged = a.pairs <= kGroupLdsWeights ? ids * 3u : a.pairs <= kGroupLdsPairs ? ids : 0u;
    // four runs where one would take several steps of loads and of placement (a workgroup of 1,024 starts later than one of 256)
    if (a.pairs > 2048u) hipLaunchKernelGGL(k_group<4>, grid, dim3(1024), 4u * SHRIKE_MAX_ROUTER_EXPERTS * 4u + staged, s, a);
    else hipLaunchKernelGGL(k_group<1>, grid, dim3(256), SHRIKE_MAX_ROUTER_EXPERTS * 4u + staged, s, a);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

int shrike_hip_shared_scalar_gate_rows(void *stream, const shrike_projection *gate_row, uint32_t meta_dtype, const void *d_x,
                                       uint32_t x_stride_elements, void *d_gate, uint32_t rows, uint32_t d) {
    SHRIKE_REQUIRE(gate_row && gate_row->weights && gate_row->scales && gate_row->biases, "scalar gate rows: the gate row must be bound");
    SHRIKE_REQUIRE(d_x && d_gate, "scalar gate rows: NULL buffer");
    // Elementwise.swift:148
    SHRIKE_REQUIRE(d > 0 && d % SHRIKE_GROUP_SIZE == 0, "shared_scalar_gate_rows drops the tail unless d is a multiple of 64");
    SHRIKE_REQUIRE(x_stride_elements >= d && x_stride_elements % 2u == 0, "scalar gate rows: x stride is too small or odd");
    SHRIKE_REQUIRE(meta_dtype <= SHRIKE_META_F16, "scalar gate rows: metaDtype=%u is not a known value", meta_dtype);
    if (rows == 0) return 0;
    auto launch = [&](auto kernel, uint32_t of_workgroup) {
        hipLaunchKernelGGL(kernel, dim3((rows + of_workgroup - 1u) / of_workgroup), dim3(256), 0, as_stream(stream),
                           static_cast<const uint8_t *>(gate_row->weights), static_cast<const uint16_t *>(gate_row->scales),
                           static_cast<const uint16_t *>(gate_row->biases), meta_dtype, static_cast<const uint16_t *>(d_x),
                           x_stride_elements, static_cast<uint16_t *>(d_gate), d, rows);
    };
    // (a row and four a workgroup, rows of 2,048: 1,000 rows 3.0 and 3.2 us, 2,048 4.2 and 3.4, 4,096 5.8 and 4.1; two: 4.4)
    if (rows >= 2048u) launch(k_scalar_gate_rows<4>, 4u);
    else launch(k_scalar_gate_rows<1>, 1u);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

int shrike_hip_sigmoid_scalar_mul_rows(void *stream, void *d_y, const void *d_gate, uint32_t d, uint32_t rows) {
    SHRIKE_REQUIRE(d_y && d_gate, "sigmoid scalar mul rows: NULL buffer");
    SHRIKE_REQUIRE(d % 8u == 0 && reinterpret_cast<uintptr_t>(d_y) % 16u == 0, "sigmoid scalar mul rows: d must be a multiple of 8 and y 16-byte aligned");
    const uint64_t slots = uint64_t(rows) * (d / 8u);
    if (slots == 0) return 0;
    hipLaunchKernelGGL(k_sigmoid_scalar_mul_rows, dim3(uint32_t((slots + 255u) / 256u)), dim3(256), 0, as_stream(stream),
                       static_cast<uint16_t *>(d_y), static_cast<const uint16_t *>(d_gate), d, rows);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

int shrike_hip_prefill_reduce(void *stream, const void *d_route_partials, const void *d_route_weights, void *d_h2,
                              uint32_t query_count, uint32_t top_k, uint32_t d) {
    SHRIKE_REQUIRE(d_route_partials && d_route_weights && d_h2, "prefill reduce: NULL buffer");
    SHRIKE_REQUIRE(d % 8u == 0 && top_k > 0, "prefill reduce: D must be a multiple of 8 and topK positive");
    const size_t slots = size_t(query_count) * (d / 8u);
    if (slots == 0) return 0;
    hipLaunchKernelGGL(k_prefill_reduce, dim3(uint32_t((slots + 255u) / 256u)), dim3(256), 0, as_stream(stream),
                       static_cast<const uint16_t *>(d_route_partials), static_cast<const uint16_t *>(d_route_weights),
                       static_cast<uint16_t *>(d_h2), query_count, top_k, d);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

int shrike_hip_residual_add_f16(void *stream, void *d_hidden, const void *d_delta, uint64_t count) {
    SHRIKE_REQUIRE(d_hidden && d_delta, "residual add: NULL buffer");
    SHRIKE_REQUIRE((reinterpret_cast<uintptr_t>(d_hidden) | reinterpret_cast<uintptr_t>(d_delta)) % 16u == 0,
                   "residual add: buffers must be 16-byte aligned");
    if (count == 0) return 0;
    const uint64_t threads = (count + 7u) / 8u;
    hipLaunchKernelGGL(k_residual_add, dim3(uint32_t((threads + 255u) / 256u)), dim3(256), 0, as_stream(stream),
                       static_cast<uint16_t *>(d_hidden), static_cast<const uint16_t *>(d_delta), count);
    SHRIKE_HIP(hipGetLastError());
    return 0;
}

}  // extern "C"
