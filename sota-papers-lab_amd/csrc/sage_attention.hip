// SageAttention2 attention kernel for gfx950 (CDNA4 MFMA, wave64).
//
// Semantics follow sezer-muhammed/sota-papers-lab,
// platform/spl-nn/cuda/sage_attn.cu:135-424 (sg_attn<false>): INT8 Q K^T with
// int32 accumulation and the dequant scale q_scale * k_scale folded into the
// exp2 argument, an online softmax in log2 units, P = 448 * 2^(x - m) rounded
// to E4M3, an FP8 P.V with fp32 accumulation, out = O / l * v_scale + v_mean.
// The layout is this build's own, designed for CDNA4:
//
// - One workgroup = 4 wave64s = 128 queries of one (batch, head); each wave
//   owns 32 queries and walks the keys in 64-key blocks.
// - The wave computes S^T = K Q^T with v_mfma_i32_32x32x32_i8: Q^T is the B
//   operand and stays in registers for the whole sweep; K is the A operand,
//   read from LDS. In the 32x32 accumulator a lane holds ONE query (its
//   column) and 16 keys, so every softmax statistic of a query lives in one
//   lane and its partner lane (lane ^ 32): the row max and row sum need a
//   single cross-half exchange.
// - O^T = V^T P^T with v_mfma_scale_f32_32x32x64_f8f6f4 (E4M3, unit scales):
//   P^T is the B operand, built in registers straight from the S^T
//   accumulators (4 keys per register, v_cvt_pk_fp8_f32); V^T is the A
//   operand, stored by the prologue with its keys in that register order
//   (v8_position). P never goes through LDS, and the O^T accumulator again
//   holds one query per lane, so rescaling by alpha is lane-local.
// - The INT8 accumulators start from the bits of 1.5 * 2^23, so each score
//   register already holds the float 1.5 * 2^23 + S (exact for |S| < 2^22):
//   no int -> float conversions. The row max runs on those bits (positive
//   floats order like their bit patterns, v_max3_i32), and the bias comes
//   off inside the exp2 FMA through xoff = -(1.5 * 2^23) * sc, the
//   reference's default logit arithmetic (SG_FAST_EXP=1, sage_attn.cu:23-31,
//   262-300), in the same fp32 operation order.
// - O is rescaled only in blocks where some row's running max moved.
// - O accumulates on the MFMA in fp32 across blocks (O = alpha * O + P.V):
//   the MFMA adds its product to C exactly in fp32, so the reference's
//   separate per-block fp32 partial is not needed.
// - K and V tiles are double-buffered in LDS with an XOR swizzle over
//   256-byte lines (conflict-free b128 operand reads), filled by direct
//   global -> LDS loads from a uniform SGPR base (no staging registers).
// - A wave runs one block at a time (QK^T, softmax, P.V); the other waves on
//   its SIMD fill the MFMA and VALU gaps: three a SIMD at head dim 128, four
//   at head dim 64. Q^T stays in registers; at head dim 128 the K operands
//   of one 32-key sub-tile at a time make room for it.
// - Workgroups are dealt to XCDs so that the ones sharing a head's K and V
//   share an L2; causal tiles are dealt longest first across each XCD's
//   heads.
// - KV merging (MERGE, the reference's sg_attn_merge, sage_attn.cu:238-246,
//   264-305): every key carries a log2(member count) bias, staged per block
//   in LDS beside K and V. The log2 logit x = S * sc + bias is formed before
//   the row max (fmaf(1.5 * 2^23 + S, sc, fmaf(-1.5 * 2^23, sc, bias))), and
//   P = 2^(x + log2(448) - m); padding keys carry -inf and need no mask.
#include "sage_attn_device.hpp"
#include "sage_internal.hpp"

namespace sage {

// INT8 Q of a wave's 32 queries q0 .. q0 + 31 of one head (sage_quant.cu:85-127;
// the prologue's tile_q8, the same codes and scales bit for bit), in a forward
// call: the rows come from the 16-bit queries, the codes and scales go to the
// workspace and, through `stage` (32 D bytes of LDS, this wave's alone), to
// the wave's MFMA operands. Left to the prologue, Q costs it 2 bytes read and
// one written an element, and one read back here, all at the memory's rate;
// here the same bytes stream under the other workgroups' key loops, which
// leave the memory idle. sage_prep at B2 H32 N4096 D128 41 -> 29 us, grouped
// 32/8 N8192 27 -> 11; this kernel pays about 450 VALU instructions a wave and
// the rows' latency, 8 us of 331. Whole forwards: 1.4 to 3.5% faster.
// D/8 lanes hold a row, 8 channels a lane, 512/D rows at a time; rows past the
// sequence are zeros. Its first half of iterations is the first 16-row group.
template <int D>
__device__ __forceinline__ void quantise_q(const uint16_t* q, int8_t* __restrict__ q8,
                                           float* __restrict__ q_scale, const Geom& g, int q0, int lane,
                                           uint8_t* stage, v4i (&qa)[D / 32], float& qs) {
#pragma clang fp contract(off)
    constexpr int CH = D / 8, RPI = 64 / CH, NI = 32 / RPI, KCPR = D / 16;
    const int ch = lane % CH, slot = lane / CH;
    typedef unsigned nt_u4 __attribute__((ext_vector_type(4)));
    typedef unsigned nt_u2 __attribute__((ext_vector_type(2)));
    nt_u4 raw[NI];
    const uint16_t* row0 = q + (long long)(q0 + slot) * g.q_st + ch * 8;
    const long long rstep = RPI * g.q_st;
    if (q0 + 32 <= g.tokens) {
#pragma unroll
        for (int i = 0; i < NI; i++) raw[i] = __builtin_nontemporal_load(reinterpret_cast<const nt_u4*>(row0 + i * rstep));
    } else {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            raw[i] = nt_u4{0, 0, 0, 0};
            if (q0 + slot + i * RPI < g.tokens)
                raw[i] = __builtin_nontemporal_load(reinterpret_cast<const nt_u4*>(row0 + i * rstep));
        }
    }
    // Row maxima on the 16-bit magnitudes, two a register: finite bf16 and
    // fp16 magnitudes order like their bits, and anything above infinity's is
    // a NaN, which fmaxf would skip (the general path below).
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    const bool half = g.flags & F_IN_F16;
    uint32_t top[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        us2 t = {0, 0};
#pragma unroll
        for (int i = j * NI / 2; i < (j + 1) * NI / 2; i++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                t = __builtin_elementwise_max(t, __builtin_bit_cast(us2, raw[i][c] & 0x7fff7fffu));
        top[j] = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u32(max((uint32_t)t.x, (uint32_t)t.y)));
    }
    float sc[2];
    auto codes = [&](bool half, bool near, const float* amax) __attribute__((always_inline)) {
        float inv[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            inv[j] = amax[j] > 0.f ? 127.0f / amax[j] : 0.f;
            sc[j] = amax[j] * (1.0f / 127.0f) * g.q_mul;
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            float x[8];
            unpack8(make_uint4(raw[i].x, raw[i].y, raw[i].z, raw[i].w), x, half);
            const float v = inv[2 * i / NI];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = x[e] * v;
            nt_u2 w;
            w.x = near ? s8x4_near(x[0], x[1], x[2], x[3]) : s8x4(x[0], x[1], x[2], x[3]);
            w.y = near ? s8x4_near(x[4], x[5], x[6], x[7]) : s8x4(x[4], x[5], x[6], x[7]);
            const int row = slot + i * RPI;
            __builtin_nontemporal_store(w, reinterpret_cast<nt_u2*>(q8 + row * D + ch * 8));
            *reinterpret_cast<nt_u2*>(stage + 16 * swz(row * KCPR + (ch >> 1), KCPR) + 8 * (ch & 1)) = w;
        }
    };
    // One branch on the input type and range for the whole tile.
    float amax[2];
#pragma unroll
    for (int j = 0; j < 2; j++) amax[j] = half ? f16_to_f32(top[j]) : __uint_as_float(top[j] << 16);
    const uint32_t inf = half ? 0x7c00u : 0x7f80u;
    bool plain = true;  // no NaN, and 127 / amax finite (or no use made of it)
#pragma unroll
    for (int j = 0; j < 2; j++) plain = plain && top[j] <= inf && (top[j] == 0 || code_scale_ok(127.0f / amax[j]));
    if (!plain) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            amax[j] = 0.f;
            for (int i = j * NI / 2; i < (j + 1) * NI / 2; i++)
                for (int c = 0; c < 4; c++) {
                    const uint32_t w = raw[i][c];
                    const float lo = half ? f16_to_f32(w & 0xffffu) : __uint_as_float(w << 16);
                    const float hi = half ? f16_to_f32(w >> 16) : __uint_as_float(w & 0xffff0000u);
                    amax[j] = fmaxf(amax[j], fmaxf(fabsf(lo), fabsf(hi)));
                }
            amax[j] = wave_max(amax[j]);
        }
        if (half)
            codes(true, false, amax);
        else
            codes(false, false, amax);
    } else if (half) {
        codes(true, true, amax);
    } else {
        codes(false, true, amax);
    }
    if (lane < 2) q_scale[lane] = lane ? sc[1] : sc[0];
    qs = lane & 16 ? sc[1] : sc[0];
    // The wave's own LDS operations complete in order.
#pragma unroll
    for (int s = 0; s < D / 32; s++)
        qa[s] = *reinterpret_cast<const v4i*>(stage + 16 * swz((lane & 31) * KCPR + 2 * s + (lane >> 5), KCPR));
}

// Workgroups a CU: four at head dim 64 (<= 128 VGPRs), three at head dim 128
// (<= 168); the merged head-dim-128 kernel needs the registers of two.
// QF (a forward call): the workgroup quantises its own queries (quantise_q)
// instead of reading the prologue's codes, and the output may be those queries
// themselves (q_readable_beside), so neither pointer is __restrict__.
template <int D, bool CAUSAL, bool MERGE, bool QF>
__global__ __launch_bounds__(256, D == 64 ? 4 : (MERGE ? 2 : 3)) void sage_attn(const uint16_t* q, int8_t* __restrict__ q8,
                                                    float* __restrict__ q_scale,
                                                    const int8_t* __restrict__ k8,
                                                    const float* __restrict__ k_scale,
                                                    const uint8_t* __restrict__ v8, const float* __restrict__ stats,
                                                    const float* __restrict__ kbias, uint16_t* out,
                                                    Geom g) {
    constexpr int BN = ATTN_BN;
    constexpr int KS = D / 32;            // INT8 k-steps of 32 channels
    constexpr int DT = D / 32;            // 32-channel tiles of O^T
    constexpr int TILE = BN * D;          // bytes of one K tile and of one V tile
    constexpr int CPT = TILE / 16 / 256;  // 16-byte chunks per thread per tile
    constexpr int KCPR = D / 16;          // chunks per K row
    static_assert(CPT >= 1, "tile too small for 256 threads");

    // K and V are double-buffered separately: step j reads K(j) and V(j)
    // while K(j+1) and V(j+1) arrive in the other buffers. Separate LDS
    // objects let the compiler see that the direct-to-LDS prefetch into one
    // buffer never aliases the MFMA operand reads of another.
    __shared__ __attribute__((aligned(16))) uint8_t ldsK0[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsK1[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsV0[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsV1[TILE];
    // Merge biases of the current and the next block.
    __shared__ __attribute__((aligned(16))) float ldsB0[MERGE ? BN : 4];
    __shared__ __attribute__((aligned(16))) float ldsB1[MERGE ? BN : 4];
    // Merged: each wave's per-key logit offsets bias - 1.5 * 2^23 * scl of the
    // current block, for each of the two Q-scale groups of its 32 queries.
    __shared__ __attribute__((aligned(16))) float ldsC[MERGE ? 4 * 2 * BN : 4];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int ntq = gridDim.x;
    const int lin = blockIdx.x + ntq * (blockIdx.y + gridDim.y * blockIdx.z), total = ntq * gridDim.y * gridDim.z;
    int qt, hb;  // query tile; head slot b * heads + h
    if (CAUSAL && causal_longest_first(total, ntq)) {
        // XCD x holds head slots [x * hx, (x + 1) * hx); its i-th workgroup
        // takes query tile ntq - 1 - i / hx of head slot x * hx + i % hx, so
        // the XCD deals its tiles longest first across all of its heads.
        const int per = total / NUM_XCD, hx = per / ntq, x = lin % NUM_XCD;
        int i = lin / NUM_XCD;
        // Where all workgroups are resident at once, workgroup i and i + 32 of
        // an XCD share a CU (the dispatcher walks its 32 CUs), and dealt
        // longest first throughout the first CUs get the longest of every
        // batch. Reversing every other batch evens the CUs' sums (D 64 768
        // tiles N 4096 65.0 -> 58.6 us, 1024 N 16384 257 -> 234; D 128 704 N
        // 1400 40.2 -> 36.9); with more workgroups the later ones go where
        // one has ended, and the order makes no difference.
        if (per <= 32 * (D == 64 ? 4 : 3)) {
            const int b0 = i & ~31;
            if ((i & 32) == 0) i = b0 + min(32, per - b0) - 1 - (i - b0);
        }
        qt = ntq - 1 - i / hx;
        hb = x * hx + i % hx;
    } else {
        const int tile = xcd_tile(lin, total);
        qt = CAUSAL ? ntq - 1 - tile % ntq : tile % ntq;  // causal: heavy tiles of a head first
        hb = tile / ntq;
    }
    const int h = hb % g.heads, b = hb / g.heads, hk = h / g.group;
    const long long bh = (long long)b * g.heads + h, bhk = (long long)b * g.kv_heads + hk;
    const int q0 = qt * ATTN_ROWS + wave * 32;  // first query of this wave
    const int qi = q0 + col;                    // this lane's query

    int nblk = g.kblocks;
    if (CAUSAL) nblk = min(nblk, (qt * ATTN_ROWS + ATTN_ROWS - 1) / BN + 1);
    // Leading blocks no query of the workgroup needs masked: every key exists
    // and (causal) precedes the workgroup's first query. Merged padding keys
    // carry a -inf bias instead.
    int nfull = MERGE ? nblk : min(nblk, g.tk / BN);
    if (CAUSAL) nfull = min(nfull, (qt * ATTN_ROWS + 1) / BN);

    const uint8_t* kg = reinterpret_cast<const uint8_t*>(k8) + bhk * (long long)g.tk_pad * D;
    const uint8_t* vg = v8 + bhk * (long long)g.tk_pad * D;
    const float* ksc = k_scale + bhk * g.kblocks;

    // Direct global -> LDS copy of one tile. Lane `lane` of wave `wave` fills
    // physical chunk c of the tile, so it fetches the logical chunk that the
    // swizzle puts there (swz is an involution).
    // The tile base is uniform and is kept opaque, so that it stays in SGPRs
    // and each load takes it plus a 32-bit lane offset (instead of a 64-bit
    // per-lane address rebuilt every block); the LDS destination is uniform
    // as well (M0).
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    uint32_t foff[CPT][2];  // [chunk][K, V]
#pragma unroll
    for (int i = 0; i < CPT; i++) {
        foff[i][0] = 16u * (uint32_t)swz(i * 256 + wv * 64 + lane, KCPR);
        foff[i][1] = 16u * (uint32_t)swz(i * 256 + wv * 64 + lane, 4);
    }
    // The 64 merge biases of block blk: one dword a lane of wave 0.
    auto fetch_bias = [&](int blk, float* dst) __attribute__((always_inline)) {
        if (MERGE && wv == 0)
            __builtin_amdgcn_global_load_lds(kbias + blk * BN + lane, (__attribute__((address_space(3))) void*)dst, 4,
                                             0, 0);
    };
    auto fetch = [&](const uint8_t* src_base, int blk, uint8_t* dst, int which) __attribute__((always_inline)) {
        const uint8_t* tb = opaque_uniform(src_base + (long long)blk * TILE);
#pragma unroll
        for (int i = 0; i < CPT; i++) {
            const int c0 = i * 256 + wv * 64;
            opaque_vgpr(foff[i][which]);  // widened next to the load: base + zext(offset) form
            __builtin_amdgcn_global_load_lds(tb + (size_t)foff[i][which],
                                             (__attribute__((address_space(3))) void*)(dst + 16 * c0), 16, 0, 0);
        }
    };

    // Q^T operand: lane holds channels 32s + 16*half .. +15 of its query.
    v4i qa[KS];
    // The Q scale; the key loop floors its product with the K scale (SCALE_FLOOR).
    float qs;
    if constexpr (QF) {
        // The first tiles' copies fly meanwhile; the codes are staged in the
        // other two buffers.
        fetch(kg, 0, ldsK0, 0);
        fetch(vg, 0, ldsV0, 1);
        fetch_bias(0, ldsB0);
        const int w2 = __builtin_amdgcn_readfirstlane(wave);
        quantise_q<D>(q + b * g.q_sb + h * g.q_sh, q8 + (bh * g.tq_pad + q0) * D,
                      q_scale + bh * (g.tq_pad / QGROUP) + q0 / QGROUP, g, q0, lane,
                      (w2 < 2 ? ldsK1 : ldsV1) + (w2 & 1) * (TILE / 2), qa, qs);
        __builtin_amdgcn_sched_barrier(0);
    } else {
        const int8_t* qrow = q8 + (bh * g.tq_pad + qi) * D + 16 * half;
#pragma unroll
        for (int s = 0; s < KS; s++) qa[s] = *reinterpret_cast<const v4i*>(qrow + 32 * s);
        qs = q_scale[bh * (g.tq_pad / QGROUP) + (qi >> 4)];
    }
    // The Q scales of the wave's two 16-query groups (wave-uniform).
    const float qsg0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(qs), 0));
    const float qsg1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(qs), QGROUP));
    // Consume the Q loads here, before the first barrier: otherwise the
    // compiler sinks them into the key loop and waits for every outstanding
    // load there, prefetches included.
#pragma unroll
    for (int s = 0; s < KS; s++) asm volatile("" ::"v"(qa[s]));
    asm volatile("" ::"v"(qs));

    // Per-lane LDS byte offsets of the MFMA operands. K row 32t + col, chunk
    // 2ks + half sits at swz((32t + col) * KCPR + 2ks + half); 32t rows are a
    // whole number of 256-byte lines whose count is a multiple of KCPR, so
    // the XOR term does not depend on t: the sub-tile term 32t * KCPR is a
    // constant offset and only the KS chunk columns need registers. V^T row
    // 32dt + col (4 chunks a row) likewise shares row col's XOR term.
    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) koff[ks] = 16 * swz(col * KCPR + 2 * ks + half, KCPR);
    const int voff0 = 16 * swz(col * 4 + 2 * half, 4), voff1 = 16 * swz(col * 4 + 2 * half + 1, 4);

    // S^T of one block (keys 32t .. 32t + 31 in s[t]) from the K tile `kt`,
    // each accumulator starting from the 1.5 * 2^23 bias.
    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; r++) magic[r] = MAGIC_BITS;
    opaque_vgpr(magic);  // kept in VGPRs, not rebuilt before every block
    auto qk = [&](const uint8_t* kt, v16i (&s)[2]) __attribute__((always_inline)) {
        const v4i (&qb)[KS] = qa;
        if constexpr (D == 128) {
            // One 32-key sub-tile's K operands at a time: the registers this
            // saves hold the Q^T operands.
#pragma unroll
            for (int t = 0; t < 2; t++) {
                uint4 ka[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    ka[ks] = *reinterpret_cast<const uint4*>(kt + 16 * 32 * t * KCPR + koff[ks]);
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const v4i av = {(int)ka[ks].x, (int)ka[ks].y, (int)ka[ks].z, (int)ka[ks].w};
                    s[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, qb[ks], ks ? s[t] : magic, 0, 0, 0);
                }
                if (t == 0) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            uint4 ka[2][KS];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    ka[t][ks] = *reinterpret_cast<const uint4*>(kt + 16 * 32 * t * KCPR + koff[ks]);
#pragma unroll
            for (int t = 0; t < 2; t++) {
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const v4i av = {(int)ka[t][ks].x, (int)ka[t][ks].y, (int)ka[t][ks].z, (int)ka[t][ks].w};
                    s[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, qb[ks], ks ? s[t] : magic, 0, 0, 0);
                }
            }
        }
    };

    v16f o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
    // m: the row's running max (log2 units); P = 2^(x - m + log2 448).
    float m = -1.0e30f, l = 0.f;

    v8i pb = {};  // P^T operand of the block whose P.V is next

    // Softmax of block blk (scores sc, biased by 1.5 * 2^23): updates m and l,
    // writes the P^T operand into pn and returns alpha = 2^(m_old - m_new);
    // grow says whether this row's max moved.
    auto softmax = [&](int blk, v16i (&sc)[2], bool masked, v8i& pn, bool& grow, const float* bias)
                       __attribute__((always_inline)) {
        // The reference's fp32 operation order for the logits: no FMA contraction.
#pragma clang fp contract(off)
        // The logit scale q_scale * k_scale, the reference's. A masked block
        // sets scores to -inf, which the product must keep (0 * -inf is a NaN),
        // so there it is floored at SCALE_FLOOR, which changes no result but an
        // exact zero scale's; merged keys are masked by a -inf bias instead.
        const float kscf = ksc[blk];
        float scl = qs * kscf;
        if constexpr (MERGE) {
            // The logit fmaf(1.5 * 2^23 + S, scl, fmaf(-1.5 * 2^23, scl, bias)):
            // the inner term depends only on the key and the query group, so
            // lane l forms it once for key l and both groups (the same value,
            // bit for bit, that each lane of the group would form) and the
            // wave reads it back from LDS in place of the bias. A wave's LDS
            // operations run in order, so the previous block's reads are done.
            float* cw = ldsC + wv * 2 * BN;
            {
                const float bl = bias[lane];
                cw[lane] = fmaf(-MAGIC, qsg0 * kscf, bl);
                cw[BN + lane] = fmaf(-MAGIC, qsg1 * kscf, bl);
            }
            const float* cg = cw + (col >> 4) * BN;
            // Element (t, r) is key 32t + 8(r >> 2) + 4 half + (r & 3): four
            // consecutive keys a 16-byte read.
            float x[32];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 cc = *reinterpret_cast<const float4*>(cg + 32 * t + 8 * j + 4 * half);
                    const float cv[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int r = 4 * j + i;
                        x[16 * t + r] = fmaf(__int_as_float(sc[t][r]), scl, cv[i]);
                    }
                }
            // 15 three-input maxima and one two-input in a tree (the logits are
            // FMA results, so fmaxf needs no canonicalising).
            auto fmax3 = [](float a, float b, float c) __attribute__((always_inline)) {
                return fmaxf(fmaxf(a, b), c);
            };
            float f3[10];
#pragma unroll
            for (int i = 0; i < 10; i++) f3[i] = fmax3(x[3 * i], x[3 * i + 1], x[3 * i + 2]);
            float mx = fmaxf(fmax3(fmax3(f3[0], f3[1], f3[2]), fmax3(f3[3], f3[4], f3[5]), fmax3(f3[6], f3[7], f3[8])),
                             fmax3(f3[9], x[30], x[31]));
            mx = fmax_halves(mx);
            const float mnew = running_max(m, mx);
            grow = mnew > m;
            const float alpha = __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            const float off = LOG2_448 - mnew;
            float p[2][16];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) p[t][r] = __builtin_amdgcn_exp2f(x[16 * t + r] + off);
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
                const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0], p[t][r0 + 1], pn[j], false);
                pn[j] = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0 + 2], p[t][r0 + 3], lo, true);
            }
            return alpha;
        }
        if (masked) {
            // Keys past the sequence, and keys after the query when causal. Element
            // (t, r) is key blk*BN + 4*half + c with the constant c below, so one
            // per-lane limit decides every element.
            const int ln = D == 128 ? lane_now() : lane, hf = ln >> 5;
            int lim = g.tk - blk * BN - 4 * hf;
            if (CAUSAL) lim = min(lim, q0 + (ln & 31) - blk * BN - 4 * hf + 1);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (32 * t + 8 * (r >> 2) + (r & 3) >= lim) sc[t][r] = NEG_INF_BITS;
            scl = fmaxf(scl, SCALE_FLOOR);
        }
        const float xoff = -MAGIC * scl;
        // Row max over this lane's 32 keys (a v_max3 tree), then the partner half.
        // 32 scores in 15 three-input maxima and one two-input: 10 over 30
        // scores, 4 over those and the last two scores, then 1 + 1.
        auto max3 = [](int a, int b, int c) __attribute__((always_inline)) { return max(max(a, b), c); };
        int m3[10];
#pragma unroll
        for (int i = 0; i < 10; i++)
            m3[i] = max3(sc[(3 * i) >> 4][(3 * i) & 15], sc[(3 * i + 1) >> 4][(3 * i + 1) & 15],
                         sc[(3 * i + 2) >> 4][(3 * i + 2) & 15]);
        const int m9 = max3(m3[0], m3[1], m3[2]), m10 = max3(m3[3], m3[4], m3[5]);
        const int m11 = max3(m3[6], m3[7], m3[8]), m12 = max3(m3[9], sc[1][14], sc[1][15]);
        int mx = max(max3(m9, m10, m11), m12);
        mx = max_halves(mx);

        // The running max in log2 units (a fully masked block gives -inf,
        // which leaves m alone); the row's largest score maps to P = 448.
        const float mnew = running_max(m, fmaf(__int_as_float(mx), scl, xoff));
        grow = mnew > m;
        const float alpha = __builtin_amdgcn_exp2f(m - mnew);
        m = mnew;

        // P = 2^(x sc + off) of the biased scores; a masked one is -inf, so
        // (scl > 0) its exp2 is 0.
        const float off = (LOG2_448 - mnew) + xoff;
        float p[2][16];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) p[t][r] = __builtin_amdgcn_exp2f(fmaf(__int_as_float(sc[t][r]), scl, off));
        // Row sum as a pairwise tree.
        float q16[16];
#pragma unroll
        for (int r = 0; r < 16; r++) q16[r] = p[0][r] + p[1][r];
#pragma unroll
        for (int w = 8; w > 0; w >>= 1)
#pragma unroll
            for (int r = 0; r < w; r++) q16[r] += q16[r + w];
        l = fmaf(l, alpha, q16[0]);

        // P^T operand: register j holds keys of accumulators 4(j%4)..+3 of
        // sub-tile j/4 (both halves are rewritten, so the register's previous
        // value serves as the unused input half and needs no zeroing).
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int t = j >> 2, r0 = 4 * (j & 3);
            const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0], p[t][r0 + 1], pn[j], false);
            pn[j] = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0 + 2], p[t][r0 + 3], lo, true);
        }
        return alpha;
    };
    // O *= alpha, only when some row of the wave moved its max.
    auto rescale = [&](float alpha, bool grow) __attribute__((always_inline)) {
        if (__any(grow)) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
    };
    // O^T += V^T P^T; V^T operands (row = channel, 4 chunks per 64-byte row)
    // read two channel tiles at a time.
    auto pv = [&](const uint8_t* vt, const v8i& pbx) __attribute__((always_inline)) {
#pragma unroll
        for (int d2 = 0; d2 < DT; d2 += 2) {
            uint4 va[2][2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                va[e][0] = *reinterpret_cast<const uint4*>(vt + 16 * 128 * (d2 + e) + voff0);
                va[e][1] = *reinterpret_cast<const uint4*>(vt + 16 * 128 * (d2 + e) + voff1);
            }
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const v8i av = {(int)va[e][0].x, (int)va[e][0].y, (int)va[e][0].z, (int)va[e][0].w,
                                (int)va[e][1].x, (int)va[e][1].y, (int)va[e][1].z, (int)va[e][1].w};
                o[d2 + e] =
                    __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pbx, o[d2 + e], 0, 0, 0, 127, 0, 127);
            }
        }
    };
    // One whole block, unpipelined: softmax, rescale, P.V.
    auto softmax_pv = [&](int blk, v16i (&sc)[2], const uint8_t* v_cur, const float* b_cur)
                          __attribute__((always_inline)) {
        bool grow;
        const float alpha = softmax(blk, sc, blk >= nfull, pb, grow, b_cur);
        __builtin_amdgcn_sched_barrier(0);
        rescale(alpha, grow);
        pv(v_cur, pb);
    };

    v16i S0[2];
    // Step j: prefetch K(j+1) and V(j+1) into the other buffers, then
    // QK^T, softmax and P.V of block j; the other waves on the SIMD fill the
    // MFMA and VALU gaps.
    auto step = [&](int blk, const uint8_t* k_cur, uint8_t* k_fill, const uint8_t* v_cur, uint8_t* v_fill,
                    const float* b_cur, float* b_fill) __attribute__((always_inline)) {
        if (blk + 1 < nblk) {
            fetch(kg, blk + 1, k_fill, 0);
            fetch(vg, blk + 1, v_fill, 1);
            fetch_bias(blk + 1, b_fill);
        }
        qk(k_cur, S0);
        softmax_pv(blk, S0, v_cur, b_cur);
        __syncthreads();
    };
    if constexpr (!QF) {
        fetch(kg, 0, ldsK0, 0);
        fetch(vg, 0, ldsV0, 1);
        fetch_bias(0, ldsB0);
    }
    __syncthreads();
    for (int blk = 0; blk < nblk; blk += 2) {
        step(blk, ldsK0, ldsK1, ldsV0, ldsV1, ldsB0, ldsB1);
        if (blk + 1 < nblk) step(blk + 1, ldsK1, ldsK0, ldsV1, ldsV0, ldsB1, ldsB0);
    }

    // out = O / l * v_scale + v_mean; lane holds channels 32dt + 8j + 4*half + 0..3.
    const float lt = sum_halves(l);
    const float inv = 1.0f / lt;
    const int ln_e = (D == 128 || MERGE) ? lane_now() : lane, half_e = ln_e >> 5, qi_e = q0 + (ln_e & 31);
    if (qi_e < g.tokens) {
        const float* vmean = stats + bhk * 4 * D + D;
        const float* vscale = vmean + D;
        uint16_t* orow = out + b * g.o_sb + (long long)qi_e * g.o_st + h * g.o_sh;
        // Pairs of outputs go through gfx950's packed converters
        // (v_cvt_pk_bf16_f32, v_cvt_pk_f16_f32: round to nearest even), one
        // uniform branch on the output type.
        // The output may be Q, so the compiler moves no load over a store: the
        // statistics of two groups of four channels are loaded ahead of their two
        // stores. One group at a time a one-block tile waited out sixteen loads at
        // head dim 128 (7.8 us, 6.4 in twos, 6.0 in fours); in fours the loads and
        // stores of a full chip's tiles crowd (2 x 4096 tokens, us a forward: 409 /
        // 410 / 414, 700 heads of 200 88.2 / 89.2 / 90.5).
        auto emit = [&](auto pack) __attribute__((always_inline)) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int j0 = 0; j0 < 4; j0 += 2) {
                    float4 vs[2], vm[2];
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int d0 = 32 * dt + 8 * (j0 + i) + 4 * half_e;
                        vs[i] = *reinterpret_cast<const float4*>(vscale + d0);
                        vm[i] = *reinterpret_cast<const float4*>(vmean + d0);
                    }
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int r = 4 * (j0 + i);
                        uint2 w;
                        w.x = pack(fmaf(o[dt][r] * inv, vs[i].x, vm[i].x), fmaf(o[dt][r + 1] * inv, vs[i].y, vm[i].y));
                        w.y = pack(fmaf(o[dt][r + 2] * inv, vs[i].z, vm[i].z), fmaf(o[dt][r + 3] * inv, vs[i].w, vm[i].w));
                        *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * (j0 + i) + 4 * half_e) = w;
                    }
                }
        };
        if (g.flags & F_OUT_F16)
            emit([](float a, float b) { return pack_f16x2(a, b); });
        else
            emit([](float a, float b) { return pack_bf16x2(a, b); });
    }
}

#ifndef SAGE_ATTN_MERGED
// Dense and causal, eight waves a workgroup: score waves and output waves
// (the layout of Tile { warps: 8, .. }).
//
// An 8-wave workgroup owns 128 queries of one (batch, head). Waves 0-3, the
// score waves, run QK^T and the online softmax of 32 queries each; waves 4-7,
// the output waves, hold the O^T accumulators of the same queries (wave
// w + 4 those of wave w) and run the rescale and P.V. The dispatcher places a
// workgroup's waves round-robin over the CU's four SIMDs, so waves w and
// w + 4 share a SIMD, and with two workgroups a CU (<= 128 VGPRs) every SIMD
// runs two score waves and two output waves: a score wave's chain is QK^T
// and softmax only, and the FP8 P.V MFMAs run under the softmax.
//
// Step j runs the softmax of block j on the score waves and the P.V of block
// j - 1 on the output waves. A score wave hands each block's P^T operand (32
// bytes a lane, the register layout of the MFMA's B operand) and its
// per-query alpha to the output wave's same lane through LDS, double-buffered
// like K and V; the V ring runs one block behind the K ring. One barrier a
// step. The arithmetic is sage_attn<D, CAUSAL, false>'s, operation for
// operation (the same logits, running max, P codes, row sums, rescale and
// accumulation order), so the outputs are bit-identical to it. It runs two
// query groups a SIMD where sage_attn runs three (head dim 128) or four (64),
// and is the slower of the two on MI355X; the default tiles select sage_attn.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(512, 2) void sage_attn_split(const int8_t* __restrict__ q8,
                                                          const float* __restrict__ q_scale,
                                                          const int8_t* __restrict__ k8,
                                                          const float* __restrict__ k_scale,
                                                          const uint8_t* __restrict__ v8,
                                                          const float* __restrict__ stats,
                                                          uint16_t* __restrict__ out, Geom g) {
    constexpr int BN = ATTN_BN, KS = D / 32, DT = D / 32, TILE = BN * D, KCPR = D / 16;
    // 16-byte chunks a K or V tile: 512 at head dim 128 (one a thread), 256 at
    // 64 (one a thread of four waves: score waves copy K, output waves V).
    constexpr int CHUNKS = TILE / 16;
    static_assert(CHUNKS == 512 || CHUNKS == 256, "head dim 64 or 128");

    __shared__ __attribute__((aligned(16))) uint8_t ldsK0[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsK1[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsV0[TILE];
    __shared__ __attribute__((aligned(16))) uint8_t ldsV1[TILE];
    // P^T operands of one block, [group][register half][lane] 16 bytes (a
    // lane's two b128 accesses are 1 KB apart, conflict-free), and alpha
    // [group][lane], double-buffered; the final row sums [group][lane].
    __shared__ __attribute__((aligned(16))) uint4 ldsP0[4 * 2 * 64];
    __shared__ __attribute__((aligned(16))) uint4 ldsP1[4 * 2 * 64];
    __shared__ __attribute__((aligned(16))) float ldsA0[4 * 64];
    __shared__ __attribute__((aligned(16))) float ldsA1[4 * 64];
    __shared__ __attribute__((aligned(16))) float ldsL[4 * 64];

    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wv & 3;
    const int ntq = gridDim.x;
    const int lin = blockIdx.x + ntq * (blockIdx.y + gridDim.y * blockIdx.z), total = ntq * gridDim.y * gridDim.z;
    int qt, hb;  // query tile; head slot b * heads + h (the same dealing as sage_attn)
    if (CAUSAL && causal_longest_first(total, ntq)) {
        const int per = total / NUM_XCD, hx = per / ntq, x = lin % NUM_XCD, i = lin / NUM_XCD;
        qt = ntq - 1 - i / hx;
        hb = x * hx + i % hx;
    } else {
        const int tile = xcd_tile(lin, total);
        qt = CAUSAL ? ntq - 1 - tile % ntq : tile % ntq;
        hb = tile / ntq;
    }
    const int h = hb % g.heads, b = hb / g.heads, hk = h / g.group;
    const long long bh = (long long)b * g.heads + h, bhk = (long long)b * g.kv_heads + hk;
    const int q0 = qt * ATTN_ROWS + grp * 32;  // first query of this wave's group

    int nblk = g.kblocks;
    if (CAUSAL) nblk = min(nblk, (qt * ATTN_ROWS + ATTN_ROWS - 1) / BN + 1);
    int nfull = min(nblk, g.tk / BN);
    if (CAUSAL) nfull = min(nfull, (qt * ATTN_ROWS + 1) / BN);

    const uint8_t* kg = reinterpret_cast<const uint8_t*>(k8) + bhk * (long long)g.tk_pad * D;
    const uint8_t* vg = v8 + bhk * (long long)g.tk_pad * D;

    // Direct global -> LDS copies of 16-byte chunks: wave slot `sl` fills
    // chunks 64 sl .. 64 sl + 63 of a tile (they land contiguously at M0;
    // lane `lane` fetches the logical chunk the swizzle puts there).
    const int sl = CHUNKS == 512 ? wv : (wv & 3);
    const uint32_t fk = 16u * (uint32_t)swz(sl * 64 + lane, KCPR), fv = 16u * (uint32_t)swz(sl * 64 + lane, 4);
    auto fetch = [&](const uint8_t* src_base, int blk, uint8_t* dst, uint32_t off) __attribute__((always_inline)) {
        const uint8_t* tb = opaque_uniform(src_base + (long long)blk * TILE);
        opaque_vgpr(off);
        __builtin_amdgcn_global_load_lds(tb + (size_t)off,
                                         (__attribute__((address_space(3))) void*)(dst + 16 * 64 * sl), 16, 0, 0);
    };
    const bool copies_k = CHUNKS == 512 || wv < 4, copies_v = CHUNKS == 512 || wv >= 4;
    // Step j's copies: K(j + 1) for the next step's QK^T, V(j) for the next
    // step's P.V.
    auto prefetch = [&](int j, uint8_t* k_fill, uint8_t* v_fill) __attribute__((always_inline)) {
        if (copies_k && j + 1 < nblk) fetch(kg, j + 1, k_fill, fk);
        if (copies_v && j < nblk) fetch(vg, j, v_fill, fv);
    };

    if (copies_k) fetch(kg, 0, ldsK0, fk);
    __syncthreads();

    if (wv < 4) {
        // ---- score wave: QK^T, online softmax, P^T and alpha to LDS ----
        const int qi = q0 + col;
        v4i qa[KS];
        {
            const int8_t* qrow = q8 + (bh * g.tq_pad + qi) * D + 16 * half;
#pragma unroll
            for (int s = 0; s < KS; s++) qa[s] = *reinterpret_cast<const v4i*>(qrow + 32 * s);
        }
        const float qs = q_scale[bh * (g.tq_pad / QGROUP) + (qi >> 4)];
#pragma unroll
        for (int s = 0; s < KS; s++) asm volatile("" ::"v"(qa[s]));
        asm volatile("" ::"v"(qs));
        const float* ksc = k_scale + bhk * g.kblocks;
        int koff[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) koff[ks] = 16 * swz(col * KCPR + 2 * ks + half, KCPR);
        v16i magic;
#pragma unroll
        for (int r = 0; r < 16; r++) magic[r] = MAGIC_BITS;
        opaque_vgpr(magic);
        float m = -1.0e30f, l = 0.f;

        auto block = [&](int blk, const uint8_t* kt, uint4* pdst, float* adst) __attribute__((always_inline)) {
            // The reference's fp32 operation order for the logits: no FMA contraction.
#pragma clang fp contract(off)
            // S^T of the block, keys 32t .. 32t + 31 in sc[t], from 1.5 * 2^23:
            // a sub-tile's four K operand reads in one LDS round trip, then its
            // four MFMAs.
            v16i sc[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                uint4 ka[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    ka[ks] = *reinterpret_cast<const uint4*>(kt + 16 * 32 * t * KCPR + koff[ks]);
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const v4i av = {(int)ka[ks].x, (int)ka[ks].y, (int)ka[ks].z, (int)ka[ks].w};
                    sc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, qa[ks], ks ? sc[t] : magic, 0, 0, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x100, KS, 0);  // the four LDS reads
                __builtin_amdgcn_sched_group_barrier(0x008, KS, 0);  // then the four MFMAs
            }
            // The logit scale, floored in masked blocks only (as sage_attn).
            float scl = qs * ksc[blk];
            if (blk >= nfull) {
                // Padding keys, and keys after the query when causal (as sage_attn).
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
            const float xoff = -MAGIC * scl;
            auto max3 = [](int a, int b, int c) __attribute__((always_inline)) { return max(max(a, b), c); };
            int m3[10];
#pragma unroll
            for (int i = 0; i < 10; i++)
                m3[i] = max3(sc[(3 * i) >> 4][(3 * i) & 15], sc[(3 * i + 1) >> 4][(3 * i + 1) & 15],
                             sc[(3 * i + 2) >> 4][(3 * i + 2) & 15]);
            const int m9 = max3(m3[0], m3[1], m3[2]), m10 = max3(m3[3], m3[4], m3[5]);
            const int m11 = max3(m3[6], m3[7], m3[8]), m12 = max3(m3[9], sc[1][14], sc[1][15]);
            int mx = max(max3(m9, m10, m11), m12);
            mx = max_halves(mx);
            const float mnew = running_max(m, fmaf(__int_as_float(mx), scl, xoff));
            const float alpha = __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            const float off = (LOG2_448 - mnew) + xoff;
            float p[2][16];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) p[t][r] = __builtin_amdgcn_exp2f(fmaf(__int_as_float(sc[t][r]), scl, off));
            float q16[16];
#pragma unroll
            for (int r = 0; r < 16; r++) q16[r] = p[0][r] + p[1][r];
#pragma unroll
            for (int w = 8; w > 0; w >>= 1)
#pragma unroll
                for (int r = 0; r < w; r++) q16[r] += q16[r + w];
            l = fmaf(l, alpha, q16[0]);
            v8i pn;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int t = j >> 2, r0 = 4 * (j & 3);
                const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0], p[t][r0 + 1], 0, false);
                pn[j] = __builtin_amdgcn_cvt_pk_fp8_f32(p[t][r0 + 2], p[t][r0 + 3], lo, true);
            }
            pdst[lane] = make_uint4((uint32_t)pn[0], (uint32_t)pn[1], (uint32_t)pn[2], (uint32_t)pn[3]);
            pdst[64 + lane] = make_uint4((uint32_t)pn[4], (uint32_t)pn[5], (uint32_t)pn[6], (uint32_t)pn[7]);
            adst[lane] = alpha;
            if (blk == nblk - 1) ldsL[grp * 64 + lane] = l;
        };
        for (int j = 0; j <= nblk; j += 2) {
            prefetch(j, ldsK1, ldsV0);
            if (j < nblk) block(j, ldsK0, ldsP0 + grp * 128, ldsA0 + grp * 64);
            __syncthreads();
            if (j + 1 <= nblk) {
                prefetch(j + 1, ldsK0, ldsV1);
                if (j + 1 < nblk) block(j + 1, ldsK1, ldsP1 + grp * 128, ldsA1 + grp * 64);
                __syncthreads();
            }
        }
    } else {
        // ---- output wave: rescale O by alpha, O^T += V^T P^T, epilogue ----
        v16f o[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
        const int voff0 = 16 * swz(col * 4 + 2 * half, 4), voff1 = 16 * swz(col * 4 + 2 * half + 1, 4);
        auto block = [&](const uint8_t* vt, const uint4* psrc, const float* asrc) __attribute__((always_inline)) {
            const float alpha = asrc[lane];
            const uint4 p0 = psrc[lane], p1 = psrc[64 + lane];
            uint4 va[DT][2];
#pragma unroll
            for (int d = 0; d < DT; d++) {
                va[d][0] = *reinterpret_cast<const uint4*>(vt + 16 * 128 * d + voff0);
                va[d][1] = *reinterpret_cast<const uint4*>(vt + 16 * 128 * d + voff1);
            }
            // alpha is exactly 1 in every row whose max did not move (the exp2
            // of 0) and below 1 otherwise; multiplying by 1 changes nothing, so
            // this is sage_attn's rescale.
            if (__any(alpha < 1.0f)) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
            }
            const v8i pb = {(int)p0.x, (int)p0.y, (int)p0.z, (int)p0.w, (int)p1.x, (int)p1.y, (int)p1.z, (int)p1.w};
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const v8i av = {(int)va[d][0].x, (int)va[d][0].y, (int)va[d][0].z, (int)va[d][0].w,
                                (int)va[d][1].x, (int)va[d][1].y, (int)va[d][1].z, (int)va[d][1].w};
                o[d] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pb, o[d], 0, 0, 0, 127, 0, 127);
            }
        };
        for (int j = 0; j <= nblk; j += 2) {
            prefetch(j, ldsK1, ldsV0);
            if (j >= 1) block(ldsV1, ldsP1 + grp * 128, ldsA1 + grp * 64);  // block j - 1 (odd)
            __syncthreads();
            if (j + 1 <= nblk) {
                prefetch(j + 1, ldsK0, ldsV1);
                block(ldsV0, ldsP0 + grp * 128, ldsA0 + grp * 64);  // block j (even)
                __syncthreads();
            }
        }

        // out = O / l * v_scale + v_mean; lane holds channels 32dt + 8j + 4*half + 0..3.
        const float lt = sum_halves(ldsL[grp * 64 + lane]);
        const float inv = 1.0f / lt;
        const int qi = q0 + col;
        if (qi < g.tokens) {
            const float* vmean = stats + bhk * 4 * D + D;
            const float* vscale = vmean + D;
            uint16_t* orow = out + b * g.o_sb + (long long)qi * g.o_st + h * g.o_sh;
            auto emit = [&](auto pack) __attribute__((always_inline)) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int d0 = 32 * dt + 8 * j + 4 * half;
                        float y[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) y[r] = fmaf(o[dt][4 * j + r] * inv, vscale[d0 + r], vmean[d0 + r]);
                        uint2 w;
                        w.x = pack(y[0], y[1]);
                        w.y = pack(y[2], y[3]);
                        *reinterpret_cast<uint2*>(orow + d0) = w;
                    }
            };
            if (g.flags & F_OUT_F16)
                emit([](float a, float b) { return pack_f16x2(a, b); });
            else
                emit([](float a, float b) { return pack_bf16x2(a, b); });
        }
    }
}

template <int D, bool CAUSAL>
static hipError_t launch_split(const AttendBufs& w, const Geom& g, hipStream_t s) {
    hipLaunchKernelGGL((sage_attn_split<D, CAUSAL>), dim3(g.tq_pad / ATTN_ROWS, g.heads, g.batch), dim3(512), 0, s,
                       w.q8, w.q_scale, w.k8, w.k_scale, w.v8, w.stats, static_cast<uint16_t*>(w.out), g);
    return hipGetLastError();
}
#endif

template <int D, bool CAUSAL, bool MERGE, bool QF>
static hipError_t launch_q(const AttendBufs& w, const Geom& g, hipStream_t s) {
    hipLaunchKernelGGL((sage_attn<D, CAUSAL, MERGE, QF>), dim3(g.tq_pad / ATTN_ROWS, g.heads, g.batch), dim3(256), 0, s,
                       w.q, w.q8, w.q_scale, w.k8, w.k_scale, w.v8, w.stats, w.kbias, static_cast<uint16_t*>(w.out), g);
    return hipGetLastError();
}

template <int D, bool CAUSAL, bool MERGE>
static hipError_t launch_d(const AttendBufs& w, const Geom& g, hipStream_t s) {
    return g.flags & F_Q_LATER ? launch_q<D, CAUSAL, MERGE, true>(w, g, s) : launch_q<D, CAUSAL, MERGE, false>(w, g, s);
}

template <bool CAUSAL, bool MERGE>
static hipError_t resources_of(int head_dim, int* regs, int* spill, int* lds) {
    hipFuncAttributes a;
    const void* f = head_dim == 64 ? reinterpret_cast<const void*>(&sage_attn<64, CAUSAL, MERGE, false>)
                                   : reinterpret_cast<const void*>(&sage_attn<128, CAUSAL, MERGE, false>);
    hipError_t e = hipFuncGetAttributes(&a, f);
    if (e != hipSuccess) return e;
    *regs = a.numRegs;
    *spill = (int)a.localSizeBytes;
    *lds = (int)a.sharedSizeBytes;
    return hipSuccess;
}

// This file is compiled twice. The dense and causal kernels (this pass) take
// LLVM's iterative occupancy-keeping pre-RA scheduler and a bottom-up post-RA
// pass, which reorder their instructions only (outputs bit-identical) and are
// faster for them; the merged kernels (SAGE_ATTN_MERGED) are faster with the
// default order and are built in the second pass.
#ifndef SAGE_ATTN_MERGED

// How the keys are split (KeySplit), by the number n of 128-query tiles, their
// remainder r over whole multiples of the chip's 256 CUs, and the 64-key blocks.
// Split kernels have a workgroup per 32 or 64 queries that exist, so for them a
// ragged tile counts by its quarters (m; 25 KV heads of 308 causal tokens, 50
// heads, head dim 128: 150 tiles, 500 workgroups, 30.2 us whole, 27.9 split).
//
// Few tiles. A tile is one wave a SIMD, and a lone wave takes 1.6 times the
// chip's best time a block, so up to about n = 256 the chip is short of waves;
// four or two shares make more of them, but read K and V once per 32 queries
// instead of 128, sweep the keys' first shares twice, and leave Q's codes to
// the prologue. They pay while their workgroups are resident at once (four a
// CU at head dim 64, two at 128: 256 and 128 tiles of four shares) and, where
// the keys are long enough for the loop to outweigh the rest, a little beyond.
// One rule for every entry, so that a forward gives prepare and attend's bits:
// the figures are of forwards, whose whole-key kernels make Q's codes; prepare
// and attend (the fused projection, normed rows) put each line a little higher,
// and where the two differ it stands where neither loses more than 3%.
// A forward on the GPU, us, whole keys / split (graph replays, one box):
//   D 64        96 tiles N 684: 23.5 / 18.4          192, N 100: 17.8 / 18.3   192, N 1000: 27.6 / 25.0
//               224, N 484: 22.9 / 23.3              224, N 2020: 39.4 / 38.6  256, N 1000: 28.5 / 28.1
//   D 128       128, N 100: 23.3 / 21.6              144, N 100: 24.3 / 28.0   128, N 4068: 80.6 / 56.8
//               144, N 1000: 37.1 / 38.3             160, N 2020: 53.9 / 52.8  160, N 4068: 82.1 / 77.9
// A causal tile's keys end at its queries, so causal grids carry half the work
// and longer tails (whole / two shares / four):
//   D 64        192, N 740: 25.2 / 22.9 / 21.4       208, N 228: 19.6 / 19.3 / 19.6   312, N 740: 29.8 / 28.2 / 30.7
//               400, N 740: 31.4 / 32.7 / 33.5       400, N 1000: 37.5 / 38.9 / 35.0
//               440, N 2532: 58.1 / 56.6 / 53.7      480, N 2532: 50.9 / 50.8 / 51.0
//               480, N 3044: 62.1 / 65.6 / 63.6      459, N 3416: 71.7 / 67.1         480, N 4068: 87.9 / 77.8 / 76.0
//   D 128       126, N 356: 27.7 / 24.7 / 23.9       159: 29.3 / 28.9 / 30.4   204, N 740: 36.1 / 36.1 / 38.1
//               129 to 144, two shares: N 228 +1 to 3%, N 356 -7 to -1%, N 740 -7 to -1%
//               208, N 1636: 48.8 / 43.4 / 43.2      248, N 1000: 40.0 / 39.3 / 43.0
//               288, N 484: 36.7 / 40.9 / 42.7       288, N 2020: 70.8 / 63.7 / 66.3
//               352, N 2764: 70.8 / 66.1 / 72.8      352, N 1000: 51.6 / 53.6 / 54.6
// With fewer than five heads an XCD's range lies within one head, whose long
// tiles are all its work, so there the line is where the XCDs hold every
// workgroup at once or little more:
//   D 64 480, 2 heads (29412 keys) 415 / 457 / 418, 3 heads 279 / 280 / 297;
//   D 128 252, 4 heads 136 / 113 / 116; 278, 2 heads 297 / 379 / 304; 284, 4 heads 155 / 169 / 156.
// Merged (whole / two shares):
//   D 64        222, stride 2, 1 frame: 24.3 / 24.0  220, 8 frames: 49.9 / 45.5
//               176, stride 4, 8 frames: 40.6 / 39.2 222, stride 4, 1 frame: 32.4 / 35.2
//   D 128       120, stride 2, 1 frame: 34.7 / 30.8  170, 3 frames: 45.8 / 47.0
//               102, stride 4, 3 frames: 48.6 / 46.1 120, 1 frame: 45.3 / 49.2
//
// A few tiles over. Whole tiles alone give r CUs one tile more than the rest,
// and those set the time. Left whole beside the others split into four
// workgroups each, the remainder spreads over all CUs. Its own limit is
// residency again (three workgroups a CU at head dim 128: 64 split tiles beside
// 512 whole ones); short keys, and more whole tiles a CU, leave it less to gain
// (whole / r split):
//   D 64  r 64 over 256, N 100: 22.0 / 21.7   144, N 100: 23.5 / 24.9   176, N 484: 30.5 / 30.1   128, N 3044: 68.9 / 59.2
//         64 over 512, N 228: 30.8 / 30.2     128, N 484: 37.4 / 37.3   128, N 1000: 47.8 / 45.6   (136 is a second round)
//         32 over 768, N 228: 38.2 / 38.3     64, N 484: 45.7 / 45.2    112, N 996: 58.4 / 58.6   108, N 1508: 73.2 / 72.0
//         64 over 1024, N 484: 54.6 / 54.3    80, N 1508: 87.6 / 86.8
//         72 over 1280, N 1000: 81.7 / 83.2   64, N 1508: 102.4 / 100.8 64 over 1536, N 1000: 92.2 / 93.4, 2020: 139.6 / 137.2
//   D 128 r 64 over 256, N 100: 32.8 / 31.4   88, N 1000: 50.6 / 51.0   80, N 3044: 91.9 / 89.2   96, N 5604: 142 / 135
//         32 over 512, N 484: 56.3 / 56.7     64, N 1000: 69.6 / 68.5   72, N 1000: 69.5 / 73.4   88, N 12772: 387 / 358
//         32 over 768, N 484: 74.5 / 75.1     64, N 1000: 91.3 / 90.5   80, N 2020: 128.9 / 130.8 66, N 17764: 700 / 645
//         32 over 1024, N 3044: 200 / 195     32, N 4068: 244 / 250     56, N 3044: 200 / 213     32, N 5604: 314 / 301
//         32 over 1280, N 2020: 179.8 / 180.2 64, N 4068: 291 / 288     32 over 1536, N 2020: 207.5 / 208.5, 4068: 336 / 329
// The tile of the context's Config does not matter here: it picks a layout,
// never a result.
KeySplit key_split(int head_dim, int tokens, int heads, int kblocks, int merge, bool causal) {
    const bool wide = head_dim == 128;
    const long long n = ((long long)tokens + 127) / 128 * heads;
    // (Of a key block or three there is nothing to share.)
    const long long m = kblocks >= 4 ? (((long long)tokens + 31) / 32 * heads + 3) / 4 : n;
    if (merge > 1) return {m <= (wide ? (merge == 2 ? 128 : 104) : (merge == 2 ? 224 : 192)) ? 2 : 0, 0};
    if (causal && !wide) {
        if (kblocks < 16) return {m <= 200 ? 4 : m <= 320 ? 2 : 0, 0};
        return {m <= (kblocks >= 52 && heads >= 5 ? 480 : 448) ? 4 : 0, 0};
    }
    if (causal) {
        if (kblocks < 16) return {m <= 128 ? 4 : m <= 144 && kblocks >= 5 ? 2 : 0, 0};
        return {m <= 208 ? 4 : m <= (heads >= 5 ? 288 : 256) ? 2 : 0, 0};
    }
    if (m <= (wide ? (kblocks >= 24 ? 160 : 128) : (kblocks >= 16 ? 224 : 192))) return {4, 0};
    const long long f = n / 256, r = n % 256;
    if (f == 0 || f > 6 || r == 0) return {0, 0};
    // [whole tiles a CU - 1]: the largest remainders that are split from so many
    // key blocks on.
    struct Line {
        int most, blocks;
    };
    static constexpr Line LINES[2][6][3] = {{{{64, 1}, {96, 4}, {176, 8}},
                                             {{64, 1}, {128, 8}},
                                             {{32, 6}, {80, 8}, {112, 16}},
                                             {{64, 8}, {80, 16}},
                                             {{80, 16}},
                                             {{64, 24}}},
                                            {{{64, 1}, {96, 32}},
                                             {{64, 8}, {96, 48}},
                                             {{64, 12}, {96, 48}},
                                             {{48, 48}},
                                             {{64, 32}},
                                             {{64, 64}}}};
    for (const Line& l : LINES[wide][f - 1])
        if (r <= l.most && kblocks >= l.blocks) return {4, (int)(n - r)};
    return {0, 0};
}

static KeySplit key_split(int head_dim, const Geom& g) {
    return key_split(head_dim, g.tokens, g.heads * g.batch, g.kblocks, g.merge, g.flags & F_CAUSAL);
}

// The whole-key four-wave kernels have the variant; the sage options' QK
// LayerNorm of Q stays in the prologue.
bool attention_quantises_q(int head_dim, const Geom& g) {
    return !(g.flags & F_LN_Q) && (g.merge > 1 || !(g.flags & F_WAVES8)) && key_split(head_dim, g).shares == 0;
}

// Dense, causal (an extension) or merged (sg_attn_merge); the API refuses
// causal masking over merged keys.
hipError_t launch_attention(int head_dim, const AttendBufs& w, const Geom& g, hipStream_t s) {
    if (const KeySplit k = key_split(head_dim, g); k.shares) return launch_attention_keys(head_dim, k, w, g, s);
    if (g.merge > 1) return launch_attention_merged(head_dim, w, g, s);
    if (g.flags & F_WAVES8) {
        if (head_dim == 64)
            return (g.flags & F_CAUSAL) ? launch_split<64, true>(w, g, s) : launch_split<64, false>(w, g, s);
        return (g.flags & F_CAUSAL) ? launch_split<128, true>(w, g, s) : launch_split<128, false>(w, g, s);
    }
    if (head_dim == 64)
        return (g.flags & F_CAUSAL) ? launch_d<64, true, false>(w, g, s) : launch_d<64, false, false>(w, g, s);
    return (g.flags & F_CAUSAL) ? launch_d<128, true, false>(w, g, s) : launch_d<128, false, false>(w, g, s);
}

hipError_t attention_resources(int head_dim, bool causal, bool merge, bool waves8, int* regs, int* spill, int* lds) {
    if (merge) return attention_resources_merged(head_dim, regs, spill, lds);
    if (waves8) {
        hipFuncAttributes a;
        const void* f = head_dim == 64
                            ? (causal ? reinterpret_cast<const void*>(&sage_attn_split<64, true>)
                                      : reinterpret_cast<const void*>(&sage_attn_split<64, false>))
                            : (causal ? reinterpret_cast<const void*>(&sage_attn_split<128, true>)
                                      : reinterpret_cast<const void*>(&sage_attn_split<128, false>));
        hipError_t e = hipFuncGetAttributes(&a, f);
        if (e != hipSuccess) return e;
        *regs = a.numRegs;
        *spill = (int)a.localSizeBytes;
        *lds = (int)a.sharedSizeBytes;
        return hipSuccess;
    }
    return causal ? resources_of<true, false>(head_dim, regs, spill, lds)
                  : resources_of<false, false>(head_dim, regs, spill, lds);
}

#else

hipError_t launch_attention_merged(int head_dim, const AttendBufs& w, const Geom& g, hipStream_t s) {
    return head_dim == 64 ? launch_d<64, false, true>(w, g, s) : launch_d<128, false, true>(w, g, s);
}

hipError_t attention_resources_merged(int head_dim, int* regs, int* spill, int* lds) {
    return resources_of<false, true>(head_dim, regs, spill, lds);
}

#endif

}  // namespace sage
