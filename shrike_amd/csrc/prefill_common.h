// Shared between the prefill translation units: the device row-tile table that the
// grouping kernels write and the grouped FFN reads.
#pragma once

#include "ffn_rules.h"
#include "gemv_common.h"

namespace shrike {

// fp16 halves of an fp32 value: hi + lo reproduces it to about 2^-22 relative
__device__ __forceinline__ uint32_t split_hi_lo(float v) {
    const uint16_t hi = f32_to_f16(v);
    const uint16_t lo = f32_to_f16(v - f16_to_f32(hi));
    return uint32_t(hi) | uint32_t(lo) << 16;
}

// Inclusive prefix sum over the lanes of a wave, lane 0 first; all lanes must be active. (Shifts within 16 lanes, then the last
// lanes of the rows before, each one vector operation: k_group, 32,768 pairs, 17.0 -> 15.4 us, 296 pairs 5.3 -> 4.5.)
__device__ __forceinline__ uint32_t wave_inclusive_scan_u32(uint32_t v) {
    v += dpp_u32<0x111>(v);       // row_shr 1, 2, 4, 8: nothing from beyond the row
    v += dpp_u32<0x112>(v);
    v += dpp_u32<0x114>(v);
    v += dpp_u32<0x118>(v);
    v += dpp_u32<0x142, 0xA>(v);  // row_bcast15 into rows 1 and 3
    return v + dpp_u32<0x143, 0xC>(v);  // row_bcast31 into rows 2 and 3
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    return uint32_t(__builtin_amdgcn_readlane(int(wave_inclusive_scan_u32(v)), 63));
}

// Asynchronous loads into LDS. The compiler does not know of them: the waits for them are counted by hand, and nothing
// between the first and the last of them should make it issue a vector load of its own. (One more load on its way makes a
// counted wait last longer, never end sooner, loads landing in order; but the wait for that load is for all of them. So it is
// where the loop of kWide reloads a spilled register, with 8-bit codes, twice in four groups.) The LDS address goes in m0, which the
// compiler sets as the operand it is there: a write of m0 inside the assembly would be one that it does not know of either,
// and its own uses of m0 on both sides would take each other's value for still there.
__device__ __forceinline__ void lds_load16(uint32_t lds, const void *p) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(p) : "memory");
}
// The base is moved on the scalar unit first: where the compiler has just brought it back from a vector register's lane
// (v_readlane of a spilled one), a memory instruction that reads it needs five wait states, which the compiler keeps for
// instructions that it knows and this one is not; the scalar unit waits by itself, and so does what reads its result. (The move
// stands where the wait state behind the write of m0 would.)
template <bool ONCE = false>  // ONCE: non-temporal, for whole lines only: the hint drops a line between its halves
__device__ __forceinline__ void lds_load16(uint32_t lds, const void *base, uint32_t offset) {
    const void *moved;
    if constexpr (ONCE) asm volatile("s_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0 nt" : "=&s"(moved) : "{m0}"(lds), "v"(offset), "s"(base) : "memory");
    else asm volatile("s_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(moved) : "{m0}"(lds), "v"(offset), "s"(base) : "memory");
}
// All but the wave's last COUNT loads have landed, and its reads of LDS are done.
template <int COUNT>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(COUNT) : "memory");
}
// All but the last COUNT loads have landed for every wave of the workgroup, and no wave still reads the LDS.
template <int COUNT>
__device__ __forceinline__ void wait_loads_and_sync() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(COUNT) : "memory");
}

}  // namespace shrike
