// Attention with the keys split over a workgroup's waves, for grids of too few
// query tiles to fill the chip (gfx950).
//
// sage_attn (sage_attention.hip) gives each wave 32 queries and every key: B x
// H x N / 32 waves in all. Below about two waves a SIMD that leaves SIMDs idle
// or CUs unevenly loaded, and each wave walks its blocks as one long serial
// chain (0.66 us a block at head dim 64, 1.6 times the chip's best rate). Here
// S = 4 or 2 waves share 32 queries, each taking a 1/S share of their key
// blocks: S times as many waves, each with 1/S of the chain. A workgroup is
// four waves: one query group under S = 4, two under S = 2. The HET variant
// (dense, S = 4) leaves most 128-query tiles whole, one workgroup each as in
// sage_attn, and splits the few over a whole number a CU, so that these spread
// over all CUs. key_split (sage_attention.hip) says which grids run here and
// what both sides measured: 96 tiles of 689 keys 11.8 -> 8.0 us, 128 of 8192 at
// head dim 128 118 -> 77, 352 of 2756 52.5 -> 37.4.
//
// The arithmetic is the reference's online softmax (sezer-muhammed/
// sota-papers-lab, platform/spl-nn/cuda/sage_attn.cu:135-424) with its running
// maximum: block j's probabilities are rounded to E4M3 against the maximum
// over blocks 0 .. j, not against a share's own. So a first sweep over all
// shares but the last (QK^T and the row max only, dealt evenly to the group's
// waves) gives each wave the maximum it starts from; then every wave runs its
// share as sage_attn does. The probability codes equal sage_attn's bit for
// bit; the last step adds the shares of O and l in fp32, scaled by 2^(m_w - m),
// so only that fp32 order differs from sage_attn's.
//
// K and V tiles are private to a wave: no barrier in the loop, at the price of
// reading K and V once per 32 queries. One K and one V buffer suffice: K(j + 1)
// is fetched over K(j) once QK^T has read it and lands during the softmax and
// P.V; V(j + 1) over V(j) after P.V, landing during the next QK^T and softmax.
// Four workgroups a CU at head dim 64 (registers; merged three), two at 128
// (LDS). HET at head dim 128 takes one buffer a wave for both tiles (ONE: V(j)
// over K(j), K(j + 1) over V(j), their latency left to the other waves), three
// workgroups a CU: its whole tiles fill the chip and want the waves.
#include "sage_attn_device.hpp"
#include "sage_internal.hpp"

namespace sage {

constexpr int KEY_WAVES = 4;  // waves a workgroup
constexpr int KEY_ROWS = 32;  // queries a group

// Direct global -> LDS copies and the waits that order them. A wave here keeps
// K's and V's copies in flight together and waits for the older of the two by
// its count (they complete in order). The compiler tracks its own copies
// object by object but loses that over a loop (it waited for V's copies before
// every read of K), so the copies are written out, with every wait explicit:
// nothing else in the kernel waits for them.
// The base goes through an SGPR pair that a scalar move writes inside the
// statement: a vector memory instruction may read an SGPR only five wait states
// after a vector instruction wrote it, the compiler keeps no such distance to
// an asm statement, and a base restored from a vector register's lanes
// (v_readlane) arrives right before it. A scalar read of that SGPR is
// interlocked, and a scalar write needs no wait before the load. The move is
// also the one wait state that M0, the copies' LDS base, needs before the load.
// (M0 is a reserved register that cannot be named as clobbered: a kernel that
// uses these helpers has no other use of it.)
// 4 KB, four copies of 64 lanes x 16 bytes: copy i reads base + 1024 i + even
// (odd copies: + odd) and fills dst + 1024 i + 16 lane.
__device__ __forceinline__ void copy_4k(const uint8_t* base, uint32_t even, uint32_t odd, uint32_t dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint8_t* b;
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_mov_b64 %0, %4\n\t"
        "global_load_lds_dwordx4 %2, %0\n\t"
        "global_load_lds_dwordx4 %3, %0 offset:1024\n\t"
        "global_load_lds_dwordx4 %2, %0 offset:2048\n\t"
        "global_load_lds_dwordx4 %3, %0 offset:3072"
        : "=&s"(b)
        : "s"(__builtin_amdgcn_readfirstlane((int)dst)), "v"(even), "v"(odd), "s"(base)
        : "memory");
#endif
}
// 1 KB, 16 bytes a lane.
__device__ __forceinline__ void copy_1k(const uint8_t* base, uint32_t off, uint32_t dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint8_t* b;
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_mov_b64 %0, %3\n\t"
        "global_load_lds_dwordx4 %2, %0"
        : "=&s"(b)
        : "s"(__builtin_amdgcn_readfirstlane((int)dst)), "v"(off), "s"(base)
        : "memory");
#endif
}
// 256 bytes, four a lane.
__device__ __forceinline__ void copy_256(const uint8_t* base, uint32_t off, uint32_t dst) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint8_t* b;
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_mov_b64 %0, %3\n\t"
        "global_load_lds_dword %2, %0"
        : "=&s"(b)
        : "s"(__builtin_amdgcn_readfirstlane((int)dst)), "v"(off), "s"(base)
        : "memory");
#endif
}
// At most N of the wave's vector memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_copies() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
#endif
}
// The wave's LDS reads have returned: their buffer may be refilled.
__device__ __forceinline__ void wait_reads() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
}

// The workgroup's LDS accesses so far are done; copies may still fly.
__device__ __forceinline__ void block_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}
__device__ __forceinline__ void store4(uint16_t* p, const float* y, bool f16) {
    uint2 w;
    if (f16) {
        w.x = pack_f16x2(y[0], y[1]);
        w.y = pack_f16x2(y[2], y[3]);
    } else {
        w.x = pack_bf16x2(y[0], y[1]);
        w.y = pack_bf16x2(y[2], y[3]);
    }
    *reinterpret_cast<uint2*>(p) = w;
}

// The grid of whole tiles beside split ones: 128-query tiles, dealt to the XCDs
// in contiguous ranges, of which an XCD's first whole8 are one workgroup each
// and the others four.
struct KeyGrid {
    int tiles, whole8;
};

template <int D, bool CAUSAL, bool MERGE, int S, bool HET>
__global__ __launch_bounds__(256, D == 64 ? (MERGE ? 3 : 4) : (HET ? 3 : 2)) void sage_attn_keys(
    const int8_t* __restrict__ q8, const float* __restrict__ q_scale, const int8_t* __restrict__ k8,
    const float* __restrict__ k_scale, const uint8_t* __restrict__ v8, const float* __restrict__ stats,
    const float* __restrict__ kbias, uint16_t* __restrict__ out, Geom g, KeyGrid kg8) {
    constexpr int BN = ATTN_BN, KS = D / 32, DT = D / 32, TILE = BN * D, KCPR = D / 16;
    constexpr int NL = TILE / 1024;  // 1 KB copies a tile
    constexpr bool ONE = HET && D == 128;
    __shared__ __attribute__((aligned(128))) uint8_t ldsK[KEY_WAVES * TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsV2[ONE ? 16 : KEY_WAVES * TILE];
    uint8_t* const ldsV = ONE ? ldsK : ldsV2;
    // The first sweep's maxima before shares 1 .. S - 1, [share - 1][wave][lane].
    __shared__ float ldsM[(S - 1) * KEY_WAVES * 64];
    __shared__ float ldsE[KEY_WAVES * 64];  // the running maximum after a share, [wave][lane]
    __shared__ float ldsL[KEY_WAVES * 64];  // its row sums
    // Merged: the biases of two blocks, and a block's per-key logit offsets
    // for the two Q-scale groups (as sage_attn).
    __shared__ __attribute__((aligned(16))) float ldsB[MERGE ? KEY_WAVES * 2 * BN : 4];
    __shared__ __attribute__((aligned(16))) float ldsC[MERGE ? KEY_WAVES * 2 * BN : 4];

    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    static_assert(!HET || (S == 4 && !CAUSAL && !MERGE), "whole tiles beside four shares: dense plans");
    int qt, hb;  // query tile; head slot b * heads + h
    int grp, part, q0;
    bool whole = false;
    if constexpr (HET) {
        // XCD x holds tiles [x n / 8, (x + 1) n / 8).
        const int lin = blockIdx.x, x = lin % NUM_XCD, i = lin / NUM_XCD;
        const int t0 = (int)((long long)x * kg8.tiles / NUM_XCD), cnt = (int)((long long)(x + 1) * kg8.tiles / NUM_XCD) - t0;
        const int ntq = g.q_tiles;
        whole = i < kg8.whole8;
        const int t = whole ? i : kg8.whole8 + (i - kg8.whole8) / 4, sub = (i - kg8.whole8) % 4;
        if (t >= cnt) return;
        qt = (t0 + t) % ntq;
        hb = (t0 + t) / ntq;
        grp = 0;
        part = wv;
        q0 = 128 * qt + 32 * (whole ? wv : sub);
        if (!whole && q0 >= g.tokens) return;
    } else {
        const int ntq = gridDim.x;
        const int lin = blockIdx.x + ntq * (blockIdx.y + gridDim.y * blockIdx.z), total = ntq * gridDim.y * gridDim.z;
        if (CAUSAL && causal_longest_first(total, ntq)) {
            const int per = total / NUM_XCD, hx = per / ntq, x = lin % NUM_XCD, i = lin / NUM_XCD;
            qt = ntq - 1 - i / hx;
            hb = x * hx + i % hx;
        } else {
            const int tile = xcd_tile(lin, total);
            qt = CAUSAL ? ntq - 1 - tile % ntq : tile % ntq;
            hb = tile / ntq;
        }
        grp = wv / S;
        part = wv % S;
        q0 = qt * (KEY_WAVES / S * KEY_ROWS) + grp * KEY_ROWS;
    }
    const int h = hb % g.heads, b = hb / g.heads, hk = h / g.group;
    const long long bh = (long long)b * g.heads + h, bhk = (long long)b * g.kv_heads + hk;
    const int qi = q0 + col;

    // Blocks this wave's group (a whole tile: the workgroup) attends, and
    // those of them that no query needs masked.
    const int qlo = HET && whole ? 128 * qt : q0, qhi = HET && whole ? 128 * qt + 127 : q0 + KEY_ROWS - 1;
    int nblk = g.kblocks;
    if (CAUSAL) nblk = min(nblk, qhi / BN + 1);
    int nfull = MERGE ? nblk : min(nblk, g.tk / BN);
    if (CAUSAL) nfull = min(nfull, (qlo + 1) / BN);
    // This wave's blocks (none where nblk < S and part is small).
    const int lo = part * nblk / S, hi = (part + 1) * nblk / S;

    const uint8_t* kg = reinterpret_cast<const uint8_t*>(k8) + bhk * (long long)g.tk_pad * D;
    const uint8_t* vg = v8 + bhk * (long long)g.tk_pad * D;
    const float* ksc = k_scale + bhk * g.kblocks;
    if ((whole || part == 0) && (long long)g.tk_pad * D <= WARM_BYTES)
        warm_l2<D>(kg, vg, (long long)g.tk_pad * D, q0 / 32, lds_address(ldsE + wv * 64));  // its own slot
    uint8_t* const kt = ldsK + wv * TILE;
    uint8_t* const vt = ldsV + wv * TILE;
    const uint32_t bdst = MERGE ? lds_address(ldsB + wv * 2 * BN) : 0;

    // One tile by NL copies of 64 lanes x 16 bytes; lane `lane` of copy i
    // fetches the logical chunk that the swizzle puts at chunk 64 i + lane.
    // That chunk is 64 i plus a lane term which only the parity of i changes
    // (and only for 8-chunk rows), so two lane offsets do.
    uint32_t fk[2] = {16u * (uint32_t)swz(lane, KCPR), 16u * (uint32_t)(swz(64 + lane, KCPR) - 64)};
    uint32_t fv = 16u * (uint32_t)swz(lane, 4);
    const uint32_t kdst = lds_address(kt), vdst = lds_address(vt);
    auto fetch = [&](const uint8_t* base, int blk, uint32_t dst, bool k) __attribute__((always_inline)) {
        const uint8_t* tb = base + (long long)blk * TILE;
#pragma unroll
        for (int i0 = 0; i0 < NL; i0 += 4)
            copy_4k(tb + 1024 * i0, k ? fk[0] : fv, k && D == 128 ? fk[1] : k ? fk[0] : fv, dst + 1024 * i0);
    };
    auto fetch_bias = [&](int blk, int slot) __attribute__((always_inline)) {
        if (MERGE) copy_256(reinterpret_cast<const uint8_t*>(kbias + blk * BN), 4 * lane, bdst + 256 * slot);
    };

    const int first = min(lo, nblk - 1);  // (a wave without blocks fetches one that it does not use)

    v4i qa[KS];
    {
        const int8_t* qrow = q8 + (bh * g.tq_pad + qi) * D + 16 * half;
#pragma unroll
        for (int s = 0; s < KS; s++) qa[s] = *reinterpret_cast<const v4i*>(qrow + 32 * s);
    }
    const float qs = q_scale[bh * (g.tq_pad / QGROUP) + (qi >> 4)];
    // Consumed here, so that no wait for them lands in a loop.
#pragma unroll
    for (int s = 0; s < KS; s++) asm volatile("" ::"v"(qa[s]));
    asm volatile("" ::"v"(qs));
    // The K scales of 64 blocks, one a lane: a block's is read from its lane (a
    // scalar load a block would be waited for with the LDS reads beside it).
    int kchunk = 0;
    float ksv = ksc[min(lane, g.kblocks - 1)];
    auto k_scale_of = [&](int blk) __attribute__((always_inline)) {
        if (blk >> 6 != kchunk) {
            kchunk = blk >> 6;
            ksv = ksc[min(64 * kchunk + lane, g.kblocks - 1)];
        }
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ksv), blk & 63));
    };
    const float qsg0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(qs), 0));
    const float qsg1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(qs), QGROUP));

    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) koff[ks] = 16 * swz(col * KCPR + 2 * ks + half, KCPR);
    const int voff0 = 16 * swz(col * 4 + 2 * half, 4), voff1 = 16 * swz(col * 4 + 2 * half + 1, 4);
    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; r++) magic[r] = MAGIC_BITS;
    opaque_vgpr(magic);

    auto qk = [&](const uint8_t* kp, v16i (&s)[2]) __attribute__((always_inline)) {
        uint4 ka[2][KS];
        // ONE: the operands of one row lie at koff[0] ^ 32 ks (2 ks + half is 2 ks
        // ^ half, and tiles are 128-byte aligned), so one address is kept and the
        // others are formed where they are read: kept as well, two registers
        // went to scratch memory (272 to 816 tiles of 996 to 17764 keys: 0
        // to 6.5% slower).
        [[maybe_unused]] uint32_t k0 = 0;
        if constexpr (ONE) {
            k0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)kp + (uint32_t)koff[0];
            opaque_vgpr(k0);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                if constexpr (ONE) {
#if defined(__HIP_DEVICE_COMPILE__)  // (an LDS pointer has 32 bits there)
                    typedef unsigned u4 __attribute__((ext_vector_type(4)));
                    const u4 w = *(__attribute__((address_space(3))) const u4*)((k0 ^ (uint32_t)(32 * ks)) + 16 * 32 * t * KCPR);
                    ka[t][ks] = make_uint4(w.x, w.y, w.z, w.w);
#endif
                } else {
                    ka[t][ks] = *reinterpret_cast<const uint4*>(kp + 16 * 32 * t * KCPR + koff[ks]);
                }
            }
            // (Three waves a SIMD at head dim 128: one sub-tile's operands at a time.)
            if (!ONE && t == 0) continue;
#pragma unroll
            for (int u = ONE ? t : 0; u <= t; u++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const v4i av = {(int)ka[u][ks].x, (int)ka[u][ks].y, (int)ka[u][ks].z, (int)ka[u][ks].w};
                    s[u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, qa[ks], ks ? s[u] : magic, 0, 0, 0);
                }
            if (ONE && t == 0) __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The block's logit scale; masked blocks set scores past the sequence (or
    // the query) to -inf and floor it (SCALE_FLOOR).
    auto scale_mask = [&](int blk, float kscf, v16i (&sc)[2]) __attribute__((always_inline)) {
        float scl = qs * kscf;
        if (!MERGE && blk >= nfull) {
            const int ln = lane_now(), hf = ln >> 5;
            int lim = g.tk - blk * BN - 4 * hf;
            if (CAUSAL) lim = min(lim, q0 + (ln & 31) - blk * BN - 4 * hf + 1);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (32 * t + 8 * (r >> 2) + (r & 3) >= lim) sc[t][r] = NEG_INF_BITS;
            scl = fmaxf(scl, SCALE_FLOOR);
        }
        return scl;
    };
    // Merged logits fmaf(1.5 * 2^23 + S, scl, fmaf(-1.5 * 2^23, scl, bias)) in x (as sage_attn).
    auto merged_logits = [&](int slot, float kscf, const v16i (&sc)[2], float scl, float* x) __attribute__((always_inline)) {
#pragma clang fp contract(off)
        float* cw = ldsC + wv * 2 * BN;
        const float bl = ldsB[(wv * 2 + slot) * BN + lane];
        cw[lane] = fmaf(-MAGIC, qsg0 * kscf, bl);
        cw[BN + lane] = fmaf(-MAGIC, qsg1 * kscf, bl);
        const float* cg = cw + (col >> 4) * BN;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4 cc = *reinterpret_cast<const float4*>(cg + 32 * t + 8 * j + 4 * half);
                const float cv[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
                for (int i = 0; i < 4; i++) x[16 * t + 4 * j + i] = fmaf(__int_as_float(sc[t][4 * j + i]), scl, cv[i]);
            }
    };
    // The block's row max in log2 units, over both halves of the wave.
    auto row_max = [&](const v16i (&sc)[2], float scl, const float* x) __attribute__((always_inline)) {
#pragma clang fp contract(off)
        if constexpr (MERGE) {
            auto fmax3 = [](float a, float b, float c) __attribute__((always_inline)) { return fmaxf(fmaxf(a, b), c); };
            float f3[10];
#pragma unroll
            for (int i = 0; i < 10; i++) f3[i] = fmax3(x[3 * i], x[3 * i + 1], x[3 * i + 2]);
            const float mx = fmaxf(fmax3(fmax3(f3[0], f3[1], f3[2]), fmax3(f3[3], f3[4], f3[5]), fmax3(f3[6], f3[7], f3[8])),
                                   fmax3(f3[9], x[30], x[31]));
            return fmax_halves(mx);
        } else {
            auto max3 = [](int a, int b, int c) __attribute__((always_inline)) { return max(max(a, b), c); };
            int m3[10];
#pragma unroll
            for (int i = 0; i < 10; i++)
                m3[i] = max3(sc[(3 * i) >> 4][(3 * i) & 15], sc[(3 * i + 1) >> 4][(3 * i + 1) & 15],
                             sc[(3 * i + 2) >> 4][(3 * i + 2) & 15]);
            const int m9 = max3(m3[0], m3[1], m3[2]), m10 = max3(m3[3], m3[4], m3[5]);
            const int m11 = max3(m3[6], m3[7], m3[8]), m12 = max3(m3[9], sc[1][14], sc[1][15]);
            const int mx = max_halves(max(max3(m9, m10, m11), m12));
            return fmaf(__int_as_float(mx), scl, -MAGIC * scl);
        }
    };

    float x[MERGE ? 32 : 1];
    // First sweep: the running maximum before each share's first block. The
    // group's waves take the blocks before the last share in turn, two at a
    // time (one in each buffer), so that every wave has a part of it.
    const int pre = (S - 1) * nblk / S;  // the last share's first block
    float mp[S - 1];
#pragma unroll
    for (int i = 0; i < S - 1; i++) mp[i] = -1.0e30f;
    if constexpr (ONE) {
        auto fetch1 = [&](int blk) __attribute__((always_inline)) {
            if (blk < pre) fetch(kg, blk, kdst, true);
        };
        if (!whole) {
            fetch1(part);
            for (int blk = part; blk < pre; blk += S) {
                const float kscf = k_scale_of(blk);
                wait_copies<0>();
                v16i s0[2];
                qk(kt, s0);
                wait_reads();
                fetch1(blk + S);
                const float scl = scale_mask(blk, kscf, s0);
                const float r = row_max(s0, scl, x);
#pragma unroll
                for (int i = 0; i < S - 1; i++)
                    if (blk < (i + 1) * nblk / S) mp[i] = running_max(mp[i], r);
            }
        }
    } else if (!whole) {
        auto fetch2 = [&](int blk) __attribute__((always_inline)) {
            if (blk < pre) {
                fetch_bias(blk, 0);
                fetch(kg, blk, kdst, true);
            }
            if (blk + S < pre) {
                fetch_bias(blk + S, 1);
                fetch(kg, blk + S, vdst, true);
            }
        };
        auto note = [&](int blk, float r) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < S - 1; i++)
                if (blk < (i + 1) * nblk / S) mp[i] = running_max(mp[i], r);
        };
        fetch2(part);
        for (int blk = part; blk < pre; blk += 2 * S) {
            const bool two = blk + S < pre;
            const float k0 = k_scale_of(blk), k1 = two ? k_scale_of(blk + S) : k0;
            wait_copies<0>();
            v16i s0[2], s1[2];
            qk(kt, s0);
            if (two) qk(vt, s1);
            if constexpr (MERGE) {
                // The bias slots are read before they are refilled too.
                const float scl = scale_mask(blk, k0, s0);
                merged_logits(0, k0, s0, scl, x);
                note(blk, row_max(s0, scl, x));
                if (two) {
                    const float scl1 = scale_mask(blk + S, k1, s1);
                    merged_logits(1, k1, s1, scl1, x);
                    note(blk + S, row_max(s1, scl1, x));
                }
                wait_reads();
                fetch2(blk + 2 * S);
            } else {
                wait_reads();
                fetch2(blk + 2 * S);
                const float scl = scale_mask(blk, k0, s0);
                note(blk, row_max(s0, scl, x));
                if (two) {
                    const float scl1 = scale_mask(blk + S, k1, s1);
                    note(blk + S, row_max(s1, scl1, x));
                }
            }
        }
    }
    float m = -1.0e30f;
    if (!whole) {
        fetch_bias(first, first & 1);
        fetch(kg, first, kdst, true);
        if (!ONE) fetch(vg, first, vdst, false);
#pragma unroll
        for (int i = 0; i < S - 1; i++) ldsM[(i * KEY_WAVES + wv) * 64 + lane] = mp[i];
        __syncthreads();
        // The running maximum before this wave's first block.
        if (part > 0) {
#pragma unroll
            for (int i = 0; i < S; i++) m = running_max(m, ldsM[((part - 1) * KEY_WAVES + grp * S + i) * 64 + lane]);
        }
    }

    v16i sc[2];
    v16f o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
    float l = 0.f;
    v8i pb = {};
    auto step = [&](int blk, bool more, bool shared, const uint8_t* kp, const uint8_t* vp)
                    __attribute__((always_inline)) {
        if (!shared) wait_copies<ONE ? 0 : NL>();  // K(blk) (and its bias) are in; V(blk)'s copies may still fly
        qk(kp, sc);
        if (!shared) wait_reads();
        const float kscf = k_scale_of(blk);
        if (!shared && ONE) fetch(vg, blk, kdst, false);
        if (!shared && more && !ONE) {
            fetch_bias(blk + 1, (blk + 1) & 1);
            fetch(kg, blk + 1, kdst, true);
        }
        float alpha;
        bool grow;
        {
            // The reference's fp32 operation order for the logits: no FMA contraction.
#pragma clang fp contract(off)
            const float scl = scale_mask(blk, kscf, sc);
            if constexpr (MERGE) merged_logits(blk & 1, kscf, sc, scl, x);
            const float mnew = running_max(m, row_max(sc, scl, x));
            grow = mnew > m;
            alpha = __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            const float off = MERGE ? LOG2_448 - mnew : (LOG2_448 - mnew) + -MAGIC * scl;
            float p[2][16];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    p[t][r] = __builtin_amdgcn_exp2f(MERGE ? x[MERGE ? 16 * t + r : 0] + off
                                                           : fmaf(__int_as_float(sc[t][r]), scl, off));
            float q16[16];
#pragma unroll
            for (int r = 0; r < 16; r++) q16[r] = p[0][r] + p[1][r];
#pragma unroll
            for (int w = 8; w > 0; w >>= 1)
#pragma unroll
                for (int r = 0; r < w; r++) q16[r] += q16[r + w];
            l = fmaf(l, alpha, q16[0]);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int t = j >> 2, r0 = 4 * (j & 3);
                const int lo8 = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0], p[t][r0 + 1], pb[j], false);
                pb[j] = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0 + 2], p[t][r0 + 3], lo8, true);
            }
        }
        if (__any(grow)) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
        // V(blk) is in: only K(blk + 1)'s copies were issued after it.
        if (!shared) {
            if (more && !ONE)
                wait_copies<NL + (MERGE ? 1 : 0)>();
            else
                wait_copies<0>();
        }
#pragma unroll
        for (int d2 = 0; d2 < DT; d2 += 2) {
            uint4 va[2][2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                va[e][0] = *reinterpret_cast<const uint4*>(vp + 16 * 128 * (d2 + e) + voff0);
                va[e][1] = *reinterpret_cast<const uint4*>(vp + 16 * 128 * (d2 + e) + voff1);
            }
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const v8i av = {(int)va[e][0].x, (int)va[e][0].y, (int)va[e][0].z, (int)va[e][0].w,
                                (int)va[e][1].x, (int)va[e][1].y, (int)va[e][1].z, (int)va[e][1].w};
                o[d2 + e] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pb, o[d2 + e], 0, 0, 0, 127, 0, 127);
            }
        }
        if (!shared) {
            wait_reads();
            if (more) fetch(ONE ? kg : vg, blk + 1, ONE ? kdst : vdst, ONE);
        }
    };
    if (HET && whole) {
        // Every wave has a query group of its own over all blocks, the tiles
        // shared and double-buffered (two K, two V): the copies of block j + 1
        // go out behind the barrier that follows block j - 1's last reads.
        uint8_t* const kb = ldsK;
        uint8_t* const vb = ONE ? ldsK + 2 * TILE : ldsV;
        const uint32_t kd = lds_address(kb) + 1024 * wv, vd = lds_address(vb) + 1024 * wv;
        const uint32_t fkw = 1024 * wv + (D == 128 && (wv & 1) ? fk[1] : fk[0]), fvw = 1024 * wv + fv;
        auto fetch_shared = [&](int blk) __attribute__((always_inline)) {
            const uint8_t *tk = kg + (long long)blk * TILE, *tv = vg + (long long)blk * TILE;
#pragma unroll
            for (int i = 0; i < TILE / 4096; i++) copy_1k(tk + 4096 * i, fkw, kd + (blk & 1) * TILE + 4096 * i);
#pragma unroll
            for (int i = 0; i < TILE / 4096; i++) copy_1k(tv + 4096 * i, fvw, vd + (blk & 1) * TILE + 4096 * i);
        };
        fetch_shared(0);
        for (int blk = 0; blk < nblk; blk++) {
            wait_copies<0>();
            block_barrier();
            if (blk + 1 < nblk) fetch_shared(blk + 1);
            step(blk, false, true, kb + (blk & 1) * TILE, vb + (blk & 1) * TILE);
        }
        const int lw = lane_now(), qw = q0 + (lw & 31);
        const float inv = 1.0f / sum_halves(l);
        if (qw >= g.tokens) return;
        const float* vmean = stats + bhk * 4 * D + D;
        const float* vscale = vmean + D;
        uint16_t* orow = out + b * g.o_sb + (long long)qw * g.o_st + h * g.o_sh;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d0 = 32 * dt + 8 * j + 4 * (lw >> 5);
                float y[4];
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = fmaf(o[dt][4 * j + r] * inv, vscale[d0 + r], vmean[d0 + r]);
                store4(orow + d0, y, g.flags & F_OUT_F16);
            }
        return;
    }
    if (lo < hi) {
        for (int blk = lo; blk + 1 < hi; blk++) step(blk, true, false, kt, vt);
        step(hi - 1, false, false, kt, vt);
    }

    wait_copies<0>();  // a wave without blocks has its unused tiles (and the warm-up) in flight
    // (Lane-derived values are rebuilt here rather than kept over the loop.)
    const int ln = lane_now(), qe = q0 + (ln & 31);
    // The shares of O, through the waves' own buffers (a group is four channels,
    // a lane's 16 bytes; 2 DT groups fill a buffer, so one buffer takes two
    // rounds): every wave writes its shares of a round's groups, then adds all
    // shares, in key order, of GR / S of them.
    constexpr int ROUNDS = ONE ? 2 : 1, GR = 4 * DT / ROUNDS;
    ldsE[wv * 64 + ln] = m;
    ldsL[wv * 64 + ln] = sum_halves(l);
    float f[S], inv = 0.f;
    const float* vmean = stats + bhk * 4 * D + D;
    const float* vscale = vmean + D;
    uint16_t* orow = out + b * g.o_sb + (long long)qe * g.o_st + h * g.o_sh;
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        if (r) __syncthreads();  // the last round's shares are read
#pragma unroll
        for (int i = 0; i < GR; i++) {
            const int gi = r * GR + i, dt = gi >> 2, j = gi & 3;
            *reinterpret_cast<float4*>((i < 2 * DT ? kt : vt) + (i % (2 * DT)) * 1024 + ln * 16) =
                make_float4(o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]);
        }
        __syncthreads();
        if (r == 0) {
            // m of the last share is the maximum over all keys; a wave without
            // blocks has its start (or -1e30) and zero shares.
            const float mend = ldsE[(grp * S + S - 1) * 64 + ln];
            float lt = 0.f;
#pragma unroll
            for (int i = 0; i < S; i++) {
                f[i] = __builtin_amdgcn_exp2f(ldsE[(grp * S + i) * 64 + ln] - mend);
                lt = fmaf(ldsL[(grp * S + i) * 64 + ln], f[i], lt);
            }
            inv = 1.0f / lt;
        }
#pragma unroll
        for (int e = 0; e < GR / S; e++) {
            const int i0 = part * (GR / S) + e, d0 = 8 * (r * GR + i0) + 4 * (ln >> 5);
            const uint8_t* src = (i0 < 2 * DT ? ldsK : ldsV) + grp * S * TILE + (i0 % (2 * DT)) * 1024 + ln * 16;
            float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < S; i++) {
                const float4 s = *reinterpret_cast<const float4*>(src + i * TILE);
                a[0] = fmaf(s.x, f[i], a[0]);
                a[1] = fmaf(s.y, f[i], a[1]);
                a[2] = fmaf(s.z, f[i], a[2]);
                a[3] = fmaf(s.w, f[i], a[3]);
            }
            if (qe < g.tokens) {
                float y[4];
#pragma unroll
                for (int c = 0; c < 4; c++) y[c] = fmaf(a[c] * inv, vscale[d0 + c], vmean[d0 + c]);
                store4(orow + d0, y, g.flags & F_OUT_F16);
            }
        }
    }
}

template <int D, bool CAUSAL, bool MERGE, int S>
static hipError_t launch(const AttendBufs& w, const Geom& g, hipStream_t s) {
    constexpr int ROWS = KEY_WAVES / S * KEY_ROWS;
    hipLaunchKernelGGL((sage_attn_keys<D, CAUSAL, MERGE, S, false>), dim3((g.tokens + ROWS - 1) / ROWS, g.heads, g.batch),
                       dim3(64 * KEY_WAVES), 0, s, w.q8, w.q_scale, w.k8, w.k_scale, w.v8, w.stats, w.kbias,
                       static_cast<uint16_t*>(w.out), g, KeyGrid{});
    return hipGetLastError();
}
template <int D>
static hipError_t launch_het(int whole, const AttendBufs& w, const Geom& g, hipStream_t s) {
    const int n = g.q_tiles * g.heads * g.batch, per = (n + NUM_XCD - 1) / NUM_XCD, w8 = whole / NUM_XCD;
    hipLaunchKernelGGL((sage_attn_keys<D, false, false, 4, true>), dim3(NUM_XCD * (w8 + 4 * (per - w8))),
                       dim3(64 * KEY_WAVES), 0, s, w.q8, w.q_scale, w.k8, w.k_scale, w.v8, w.stats, w.kbias,
                       static_cast<uint16_t*>(w.out), g, KeyGrid{n, w8});
    return hipGetLastError();
}

// The combinations key_split (sage_attention.hip) gives: two shares for merged
// and causal plans, four for causal and dense ones, whole tiles beside four
// shares for dense ones.
template <int D>
static hipError_t launch_d(const KeySplit& k, const AttendBufs& w, const Geom& g, hipStream_t s) {
    if (g.merge > 1) return launch<D, false, true, 2>(w, g, s);
    if (g.flags & F_CAUSAL)
        return k.shares == 4 ? launch<D, true, false, 4>(w, g, s) : launch<D, true, false, 2>(w, g, s);
    return k.whole ? launch_het<D>(k.whole, w, g, s) : launch<D, false, false, 4>(w, g, s);
}

hipError_t launch_attention_keys(int head_dim, const KeySplit& k, const AttendBufs& w, const Geom& g, hipStream_t s) {
    return head_dim == 64 ? launch_d<64>(k, w, g, s) : launch_d<128>(k, w, g, s);
}

}  // namespace sage
