// The reference's CPU expert kernel behind its own C interface: shrike_int4_affine_gemv
// (sources/ShrikeKernelsC/include/shrike_kernels.h:9-29, sources/ShrikeKernelsC/int4_affine_gemv.c:28-135)
// and CPUExpertFFN.accumulate (sources/Shrike/Kernels/CPU/CPUExpertFFN.swift:102-140), which a runner uses
// for experts it keeps in host memory. Host-only: no device call, and nothing on the GPU path calls it.
//
// out[r] = sum_g ( scale[r][g] * sum_{i in g} q[r][i] x[i]  +  bias[r][g] * sum_{i in g} x[i] ), the two
// group sums running over element pairs in order: the rounding points of the reference's portable branch
// (int4_affine_gemv.c:114-134), so that the results are its bits. A byte's two codes are widened through a
// 256-entry table; the pair sums of x do not depend on the row and are formed once a call.
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/shrike_host.h"
#include "host_common.h"

namespace {

constexpr size_t kGroupElems = SHRIKE_GROUP_SIZE, kGroupBytes = kGroupElems / 2;

struct NibblePair {
    float lo, hi;
};
struct NibbleTable {
    NibblePair of[256];
    NibbleTable() {
        for (int b = 0; b < 256; ++b) of[b] = {float(b & 0x0F), float(b >> 4)};
    }
};
const NibbleTable g_codes;

inline float bf16(uint16_t bits) {
    const uint32_t u = uint32_t(bits) << 16;
    float v;
    std::memcpy(&v, &u, sizeof v);
    return v;
}

// sum_{pairs of the group, in order} (x_even + x_odd), one value a group; the same for every row
void group_sums_of(const float *x, size_t groups, float *out) {
    for (size_t g = 0; g < groups; ++g) {
        const float *xg = x + g * kGroupElems;
        float s = 0.0f;
        for (size_t k = 0; k < kGroupBytes; ++k) s += xg[2 * k] + xg[2 * k + 1];
        out[g] = s;
    }
}

void gemv_rows_scalar(const uint8_t *weights, const uint16_t *scales, const uint16_t *biases, const float *x, const float *xsum,
                      size_t rows, size_t groups, float *out) {
    for (size_t r = 0; r < rows; ++r) {
        const uint8_t *codes = weights + r * groups * kGroupBytes;
        const uint16_t *s = scales + r * groups, *b = biases + r * groups;
        float acc = 0.0f;
        for (size_t g = 0; g < groups; ++g, codes += kGroupBytes) {
            const float *xg = x + g * kGroupElems;
            float dot = 0.0f;
            for (size_t k = 0; k < kGroupBytes; ++k) {
                const NibblePair q = g_codes.of[codes[k]];
                dot += q.lo * xg[2 * k] + q.hi * xg[2 * k + 1];
            }
            acc += bf16(s[g]) * dot + bf16(b[g]) * xsum[g];
        }
        out[r] = acc;
    }
}

#if defined(__x86_64__)

// ---- AVX-512: lane r of a vector is row r of a block of sixteen.
//
// A row's dot is one chain of additions, which bounds the scalar loop: four to five cycles a byte of codes. Side by side
// sixteen chains run in the time of one, and two blocks at once hide the addition's latency. What is left is instruction
// count, so a code is never converted: the sixteen products x * 0 ... x * 15 of one activation are a vector, formed once
// for all rows (each the very product the scalar loop forms), and a row's code picks its product by a permute, which
// reads the low four bits of its index lane alone: per sixteen rows and byte of codes two shifts, two permutes, two
// additions and 0.8 of a shuffle. One expert of 2048 x 512 (1.77 MB) on one core of an EPYC with 512-bit pipes:
// 591 us row by row (3.0 GB/s), so 82 us from the caches and 105 to 120 from DRAM (by the machine; reading the bytes and nothing
// else takes that core 38 us from DRAM, 11 from the third-level cache: the instructions bound it, not the memory); 2880 x
// 2880: 4,643 us, and 585 and 815 to 860. (Tables of eight groups, which fit the first-level cache, have every row visited in
// shorter pieces: 114 and 1,137 us from DRAM where these took 108 and 815; a table over the whole row: 126 and 793.)
#define SHRIKE_AVX512 __attribute__((target("avx512f,avx512bw,avx512vl")))

constexpr size_t kLanes = 16;
constexpr size_t kChunkGroups = 8;                   // groups whose metadata a block of rows widens at once
constexpr size_t kStretchGroups = 4 * kChunkGroups;  // groups of one table of products: 128 KB, from the second-level cache

// The 16-bit metadata of up to eight groups of a block's rows as fp32, out[g] = the rows' values of group g.
SHRIKE_AVX512 inline void widen_metadata(const uint16_t *const (&row)[kLanes], size_t groups_here, __m512 (&out)[kChunkGroups]) {
    const __mmask8 have = __mmask8((1u << groups_here) - 1u);
    __m256i v[8];  // rows i and i + 8 in the two halves
    for (int i = 0; i < 8; ++i)
        v[i] = _mm256_inserti128_si256(_mm256_castsi128_si256(_mm_maskz_loadu_epi16(have, row[i])), _mm_maskz_loadu_epi16(have, row[i + 8]), 1);
    __m256i a[8], b[8];
    for (int i = 0; i < 4; ++i) {
        a[2 * i] = _mm256_unpacklo_epi16(v[2 * i], v[2 * i + 1]);
        a[2 * i + 1] = _mm256_unpackhi_epi16(v[2 * i], v[2 * i + 1]);
    }
    for (int i = 0; i < 2; ++i) {
        b[4 * i] = _mm256_unpacklo_epi32(a[4 * i], a[4 * i + 2]);
        b[4 * i + 1] = _mm256_unpackhi_epi32(a[4 * i], a[4 * i + 2]);
        b[4 * i + 2] = _mm256_unpacklo_epi32(a[4 * i + 1], a[4 * i + 3]);
        b[4 * i + 3] = _mm256_unpackhi_epi32(a[4 * i + 1], a[4 * i + 3]);
    }
    for (int i = 0; i < 4; ++i) {
        out[2 * i] = _mm512_castsi512_ps(_mm512_slli_epi32(_mm512_cvtepu16_epi32(_mm256_unpacklo_epi64(b[i], b[i + 4])), 16));
        out[2 * i + 1] = _mm512_castsi512_ps(_mm512_slli_epi32(_mm512_cvtepu16_epi32(_mm256_unpackhi_epi64(b[i], b[i + 4])), 16));
    }
}

// One group's 32 bytes of codes of a block's rows, out[j] = the rows' word j.
SHRIKE_AVX512 inline void transpose_codes(const uint8_t *const (&row)[kLanes], size_t at, __m512i (&out)[8]) {
    __m512i v[8], a[8], b[8];  // rows i and i + 8 in the two halves
    for (int i = 0; i < 8; ++i)
        v[i] = _mm512_inserti64x4(_mm512_castsi256_si512(_mm256_loadu_si256(reinterpret_cast<const __m256i *>(row[i] + at))),
                                  _mm256_loadu_si256(reinterpret_cast<const __m256i *>(row[i + 8] + at)), 1);
    for (int i = 0; i < 4; ++i) {
        a[2 * i] = _mm512_unpacklo_epi32(v[2 * i], v[2 * i + 1]);
        a[2 * i + 1] = _mm512_unpackhi_epi32(v[2 * i], v[2 * i + 1]);
    }
    for (int i = 0; i < 2; ++i) {
        b[4 * i] = _mm512_unpacklo_epi64(a[4 * i], a[4 * i + 2]);
        b[4 * i + 1] = _mm512_unpackhi_epi64(a[4 * i], a[4 * i + 2]);
        b[4 * i + 2] = _mm512_unpacklo_epi64(a[4 * i + 1], a[4 * i + 3]);
        b[4 * i + 3] = _mm512_unpackhi_epi64(a[4 * i + 1], a[4 * i + 3]);
    }
    // quarters: b[c] holds words c (low quarter of a half) and c + 4 of rows 0-3 | 8-11, b[c + 4] of rows 4-7 | 12-15
    const __m512i low = _mm512_setr_epi64(0, 1, 8, 9, 4, 5, 12, 13), high = _mm512_setr_epi64(2, 3, 10, 11, 6, 7, 14, 15);
    for (int c = 0; c < 4; ++c) {
        out[c] = _mm512_permutex2var_epi64(b[c], low, b[c + 4]);
        out[c + 4] = _mm512_permutex2var_epi64(b[c], high, b[c + 4]);
    }
}

// BLOCKS * 16 rows against the `groups_here` groups whose products are in `table`; out carries the rows' sums from one
// stretch of groups to the next.
template <int BLOCKS>
SHRIKE_AVX512 void gemv_block(const uint8_t *weights, const uint16_t *scales, const uint16_t *biases, const float *table,
                              const float *xsum, size_t row0, size_t rows, size_t groups, size_t g0, size_t groups_here, bool first,
                              float *out) {
    const uint8_t *codes[BLOCKS][kLanes];
    __m512 s[BLOCKS][kChunkGroups], b[BLOCKS][kChunkGroups], acc[BLOCKS];
    __mmask16 live[BLOCKS];
    for (int k = 0; k < BLOCKS; ++k) {
        const uint16_t *s_row[kLanes], *b_row[kLanes];
        const size_t r0 = row0 + kLanes * size_t(k), left = rows > r0 ? rows - r0 : 0;
        live[k] = __mmask16(left >= kLanes ? 0xffffu : (1u << left) - 1u);
        for (size_t i = 0; i < kLanes; ++i) {
            const size_t r = r0 + i < rows ? r0 + i : rows - 1;  // past the last row: a copy, never stored
            codes[k][i] = weights + (r * groups + g0) * kGroupBytes;
            s_row[i] = scales + r * groups + g0;
            b_row[i] = biases + r * groups + g0;
        }
        widen_metadata(s_row, groups_here, s[k]);
        widen_metadata(b_row, groups_here, b[k]);
        acc[k] = first ? _mm512_setzero_ps() : _mm512_maskz_loadu_ps(live[k], out + r0);
    }
    // the next block's codes are asked for ahead, a line (two groups) of each row at a time: thirty-two rows are more
    // streams than the processor follows by itself (weights from DRAM: 198 us an expert of 2048 x 512 without, 108 with)
    const bool ahead = row0 + 2 * kLanes * BLOCKS <= rows;
    const size_t next = kLanes * BLOCKS * groups * kGroupBytes;
    for (size_t g = 0; g < groups_here; ++g) {
        if (ahead && g % 2 == 0)
            for (int k = 0; k < BLOCKS; ++k)
                for (size_t i = 0; i < kLanes; ++i) _mm_prefetch(reinterpret_cast<const char *>(codes[k][i] + next + g * kGroupBytes), _MM_HINT_T0);
        __m512i w[BLOCKS][8];
        __m512 dot[BLOCKS];
        for (int k = 0; k < BLOCKS; ++k) {
            transpose_codes(codes[k], g * kGroupBytes, w[k]);
            dot[k] = _mm512_setzero_ps();
        }
        const float *t = table + g * kGroupElems * kLanes;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int p = 0; p < 4; ++p, t += 2 * kLanes) {
                const __m512 even = _mm512_load_ps(t), odd = _mm512_load_ps(t + kLanes);
#pragma unroll
                for (int k = 0; k < BLOCKS; ++k) {
                    const __m512 lo = _mm512_permutexvar_ps(_mm512_srli_epi32(w[k][j], 8 * p), even);
                    const __m512 hi = _mm512_permutexvar_ps(_mm512_srli_epi32(w[k][j], 8 * p + 4), odd);
                    dot[k] = _mm512_add_ps(dot[k], _mm512_add_ps(lo, hi));
                }
            }
        }
        const __m512 xs = _mm512_set1_ps(xsum[g0 + g]);
        for (int k = 0; k < BLOCKS; ++k)
            acc[k] = _mm512_add_ps(acc[k], _mm512_add_ps(_mm512_mul_ps(s[k][g], dot[k]), _mm512_mul_ps(b[k][g], xs)));
    }
    for (int k = 0; k < BLOCKS; ++k) _mm512_mask_storeu_ps(out + row0 + kLanes * size_t(k), live[k], acc[k]);
}

SHRIKE_AVX512 void gemv_rows_avx512(const uint8_t *weights, const uint16_t *scales, const uint16_t *biases, const float *x,
                                    const float *xsum, size_t rows, size_t groups, float *table, float *out) {
    const __m512 codes = _mm512_setr_ps(0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
    for (size_t stretch = 0; stretch < groups; stretch += kStretchGroups) {
        const size_t end = groups - stretch < kStretchGroups ? groups : stretch + kStretchGroups;
        for (size_t i = stretch * kGroupElems; i < end * kGroupElems; ++i)
            _mm512_store_ps(table + (i - stretch * kGroupElems) * kLanes, _mm512_mul_ps(codes, _mm512_set1_ps(x[i])));
        for (size_t r = 0; r < rows; r += 2 * kLanes) {
            for (size_t g0 = stretch; g0 < end; g0 += kChunkGroups) {
                const size_t groups_here = end - g0 < kChunkGroups ? end - g0 : kChunkGroups;
                const float *t = table + (g0 - stretch) * kGroupElems * kLanes;
                if (rows - r > kLanes) gemv_block<2>(weights, scales, biases, t, xsum, r, rows, groups, g0, groups_here, g0 == 0, out);
                else gemv_block<1>(weights, scales, biases, t, xsum, r, rows, groups, g0, groups_here, g0 == 0, out);
            }
        }
    }
}

bool has_avx512() {
    static const bool has = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512vl");
    return has;
}

// The calling thread's table of products, from its first call to its end: 128 KB are more than a small stack of a caller's
// thread may hold, and allocated anew for every expert they may come as new pages each time. On a page boundary: eight experts
// from memory took 846 us, from the stack 861, from a table 64 bytes off one 879. Null where the processor has no AVX-512 or the
// system no memory: the rows then go one by one, to the same bits.
float *product_table() {
    struct Table {
        float *floats = nullptr;
        ~Table() { std::free(floats); }
    };
    thread_local Table table;
    if (!table.floats && has_avx512())
        table.floats = static_cast<float *>(std::aligned_alloc(4096, kStretchGroups * kGroupElems * kLanes * sizeof(float)));
    return table.floats;
}

#else

float *product_table() { return nullptr; }
void gemv_rows_avx512(const uint8_t *, const uint16_t *, const uint16_t *, const float *, const float *, size_t, size_t, float *, float *) {}

#endif

void gemv_rows(const uint8_t *weights, const uint16_t *scales, const uint16_t *biases, const float *x, const float *xsum,
               size_t rows, size_t groups, float *out) {
    // (a block costs what sixteen rows cost: a handful of rows is better off alone)
    float *table = rows >= 4 && groups > 0 ? product_table() : nullptr;
    if (table) gemv_rows_avx512(weights, scales, biases, x, xsum, rows, groups, table, out);
    else gemv_rows_scalar(weights, scales, biases, x, xsum, rows, groups, out);
}

inline float silu(float v) { return v / (1.0f + std::exp(-v)); }  // CPUExpertFFN.swift:92-94

}  // namespace

extern "C" {

void shrike_int4_affine_gemv(const uint8_t *weights, const uint16_t *scales, const uint16_t *biases, const float *x,
                             size_t rows, size_t n, float *out) {
    const size_t groups = n / kGroupElems;
    float stack_sums[64];
    std::vector<float> heap_sums;
    float *xsum = stack_sums;
    if (groups > 64) {
        heap_sums.resize(groups);
        xsum = heap_sums.data();
    }
    group_sums_of(x, groups, xsum);
    gemv_rows(weights, scales, biases, x, xsum, rows, groups, out);
}

size_t shrike_cpu_expert_ffn_scratch_floats(uint32_t d, uint32_t f) { return 2 * size_t(f) + size_t(d); }

int shrike_cpu_expert_ffn_accumulate(const void *expert, const shrike_expert_offsets *offsets, const float *x, uint32_t d,
                                     uint32_t f, float route_weight, float *scratch, float *out) {
    SHRIKE_REQUIRE(expert && offsets && x && scratch && out, "CPUExpertFFN.accumulate: NULL argument");
    SHRIKE_REQUIRE(d > 0 && f > 0 && d % kGroupElems == 0 && f % kGroupElems == 0,
                   "CPUExpertFFN.accumulate: d=%u and f=%u must be positive multiples of %u", d, f, SHRIKE_GROUP_SIZE);
    const uint8_t *base = static_cast<const uint8_t *>(expert);
    auto meta = [&](uint32_t off) { return reinterpret_cast<const uint16_t *>(base + off); };
    float *gate = scratch, *up = scratch + f, *down = scratch + 2 * size_t(f);
    // gate and up share x, and with it x's group sums (kept in the down rows' place until they are needed)
    float *xsum = down;
    group_sums_of(x, d / kGroupElems, xsum);
    gemv_rows(base + offsets->gate_w_off, meta(offsets->gate_s_off), meta(offsets->gate_b_off), x, xsum, f, d / kGroupElems, gate);
    gemv_rows(base + offsets->up_w_off, meta(offsets->up_s_off), meta(offsets->up_b_off), x, xsum, f, d / kGroupElems, up);
    for (uint32_t i = 0; i < f; ++i) gate[i] = silu(gate[i]) * up[i];
    // the activations' group sums go where `up` was
    group_sums_of(gate, f / kGroupElems, up);
    gemv_rows(base + offsets->down_w_off, meta(offsets->down_s_off), meta(offsets->down_b_off), gate, up, d, f / kGroupElems, down);
    for (uint32_t r = 0; r < d; ++r) out[r] += route_weight * down[r];
    return 0;
}

}  // extern "C"
