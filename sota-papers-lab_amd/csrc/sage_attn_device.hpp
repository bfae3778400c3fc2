// Device helpers shared by the attention kernels: score and softmax constants,
// cross-half reductions, the logit scale floor and the workgroup order.
#pragma once

#include "sage_device.hpp"

namespace sage {

constexpr int ATTN_BN = 64;  // keys per iteration (one K scale, one V block)
constexpr int MAGIC_BITS = 0x4B400000;      // bits of 1.5 * 2^23
constexpr float MAGIC = 12582912.0f;        // 1.5 * 2^23
constexpr int NEG_INF_BITS = (int)0xFF800000;  // -inf: below every biased score as an int
constexpr float LOG2_448 = 8.807354922057604f;  // P = 448 for the row max: E4M3's largest finite

// A row statistic held in lane l and its partner lane l ^ 32 (the other half
// of the wave), combined in every lane with one v_permlane32_swap of two copies
// of x: the swap's first result holds the lower half's values in both halves,
// its second the upper half's, so every lane combines the same pair in the
// same order.
__device__ __forceinline__ int max_halves(int x) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return max((int)r[0], (int)r[1]);
}
__device__ __forceinline__ float fmax_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
    // v_med3_f32 with FLT_MAX: the maximum of two non-NaN values without the
    // canonicalising v_max_f32 that fmaxf puts on each swapped register.
    return __builtin_amdgcn_fmed3f(__int_as_float((int)r[0]), __int_as_float((int)r[1]), 3.4028234663852886e38f);
}
__device__ __forceinline__ float sum_halves(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
    return __int_as_float((int)r[0]) + __int_as_float((int)r[1]);
}
// Floor of the logit scale q_scale * k_scale in masked blocks: a masked score
// is -inf and must stay -inf through the product (0 * -inf would be a NaN),
// so the product is floored where scores are masked. Below 1e-30
// the floor changes no result: every logit difference of the block is then
// under 2^22 * 1e-30 < 1e-23, far below half an ulp of the exp2 argument
// (about 8.8, ulp 2^-20), so every P and alpha come out bit-identical to the
// unfloored product's. Only an exact zero scale (an all-zero 16-row Q group,
// a K head constant over tokens) is changed: the row attends uniformly to its
// visible keys, where the reference's masked keys turn into NaNs.
constexpr float SCALE_FLOOR = 1.0e-30f;
// max(m, x) for the running max: v_med3_f32(m, x, FLT_MAX) in one instruction
// (fmaxf on the loop-carried m costs a canonicalising v_max_f32 m, m every
// block). Neither operand is a NaN: m starts at -1e30 and x is a finite logit
// or -inf.
__device__ __forceinline__ float running_max(float m, float x) {
    return __builtin_amdgcn_fmed3f(m, x, 3.4028234663852886e38f);
}
// Values the compiler may not re-derive or rematerialise: a uniform pointer
// stays in SGPRs and is not reassociated with per-lane offsets; a VGPR value
// stays where it is. (The constraints name AMDGPU register classes, so the
// statements exist only in the device pass.)
__device__ __forceinline__ const uint8_t* opaque_uniform(const uint8_t* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
    return p;
}
template <typename T>
__device__ __forceinline__ void opaque_vgpr(T& x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
}

// The dispatcher deals workgroups to the 8 XCDs round-robin by linear id,
// and each XCD has its own L2. Tile t (query tile fastest, then head, then
// batch) goes to the workgroup that gives XCD x the contiguous range of
// tiles [x * per, (x + 1) * per): the workgroups that share a head's K and V
// then read them through one L2 instead of eight. The last total % 8 tiles
// keep their place.
__device__ __forceinline__ int xcd_tile(int lin, int total) {
    const int per = total / NUM_XCD;
    if (lin >= per * NUM_XCD) return lin;
    return (lin % NUM_XCD) * per + lin / NUM_XCD;
}

// A causal query tile qt sweeps 2 qt + 2 key blocks. Dealt head by head,
// the heavy tiles of an XCD's last head start late and finish alone; dealt
// longest first across the XCD's heads, the short tiles fill the tail. That
// order needs every XCD to hold whole heads (the plain mapping above does
// then too, so the L2 sharing is unchanged).
__device__ __forceinline__ bool causal_longest_first(int total, int ntq) {
    return total % NUM_XCD == 0 && (total / NUM_XCD) % ntq == 0;
}

// This lane's index in the wave, rebuilt from v_mbcnt: values derived from the
// lane are recomputed where a rare path or the epilogue needs them instead of
// being kept live (or spilled) across the key loop.
__device__ __forceinline__ int lane_now() {
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// Brings K and V of keys 32 gi .. 32 gi + 31 of a head (kg, vg: the head's code
// arrays, `bytes` each) into this XCD's L2: one dword of every 128-byte line,
// copied to an LDS sink that nobody reads. Each 32-query group of a head calls
// it once for its own share, so a head's codes are on their way at once instead
// of a block ahead of the first wave that needs them: with few waves a SIMD a
// block takes less time than a miss. Four frames (352 tiles) 61.2 -> 58.3 us a
// forward, one frame 19.3 -> 18.8; sage_attn, whose blocks take longer, lost 2
// to 3% to it at 384 and 768 tiles. It is older than every copy that the
// caller counts, so those waits hold; the caller waits for it before it uses
// the sink's memory. Only for heads of up to WARM_BYTES of K: an XCD's 4 MB L2
// holds the K and V of the heads its workgroups are on, and a longer head's
// would be gone again before the sweep reaches them.
constexpr long long WARM_BYTES = 3LL << 19;
template <int D>
__device__ __forceinline__ void warm_l2(const uint8_t* kg, const uint8_t* vg, long long bytes, int gi, uint32_t sink) {
    const int ln = lane_now();
    const long long off = 32LL * D * gi + 128 * (ln % (D / 4));
    if (ln < D / 2 && off < bytes) {
        [[maybe_unused]] const uint8_t* p = (ln < D / 4 ? kg : vg) + off;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dword %1, off" ::"s"(__builtin_amdgcn_readfirstlane((int)sink)), "v"(p)
            : "memory");
#endif
    }
}

}  // namespace sage
